// Per-token selection (gate softmax + top-1 / top-2) shared by the routing kernels (moe_route.hip) and the
// batch-prioritised routing (moe_bpr.hip).
#pragma once
#include "scan.hpp"
#include <type_traits>
#include "../../include/lancet_hip.h"

namespace lancet {

// ---------------------------------------------------------------------------------------
// Per-token selection on the array the op is given (first max wins; slot 2 = first max with
// slot 1's expert excluded).  With logits the returned values are softmax probabilities,
// exp(x - max) / sum_e exp(x - max), the sum taken in expert order.
// Replaces the argmax / one_hot / multiply+sum micro-kernels of
// src/op/dialect/cuda/moe.cc:177-250 (three passes over [S,E] plus an [S,E] workspace).
// ---------------------------------------------------------------------------------------
// Running first-max / second-max of a row, all in scalars (no arrays, no references: the state has
// to stay in registers).  Branch-free: a lane either takes a new first choice (the old one becomes
// the second), or a new second choice, or nothing.
struct TopState {
  float v1, v2;
  int i1, i2;
};

template <int K>
__device__ __forceinline__ TopState consider(TopState t, float x, int j) {
  const bool first = (t.i1 < 0) | (x > t.v1);
  if (K == 2) {
    const bool second = !first & ((t.i2 < 0) | (x > t.v2));
    t.v2 = first ? t.v1 : (second ? x : t.v2);
    t.i2 = first ? t.i1 : (second ? j : t.i2);
  }
  t.v1 = first ? x : t.v1;
  t.i1 = first ? j : t.i1;
  return t;
}

struct Routed {
  int e0, e1;
  float p0, p1;
};

// ---- a gate row in its storage type (GD = LANCET_F32 / LANCET_BF16 / LANCET_F16), read as fp32 ----------
template <int GD>
__device__ __forceinline__ float gate_at(const void* row, int j) {
  if (GD == LANCET_F32) return static_cast<const float*>(row)[j];
  const uint32_t h = static_cast<const uint16_t*>(row)[j];
  return GD == LANCET_BF16 ? bf16_to_f32(h) : f16_to_f32(h);
}
template <int GD>
__device__ __forceinline__ float half_word(uint32_t h) {
  return GD == LANCET_BF16 ? bf16_to_f32(h) : f16_to_f32(h);
}

// the values of granule g of a row, in order
template <int GD, typename F>
__device__ __forceinline__ void walk_granule(const u32x4 x, int g, F& f) {
  if (GD == LANCET_F32) {
    f(__uint_as_float(x.x), 4 * g);
    f(__uint_as_float(x.y), 4 * g + 1);
    f(__uint_as_float(x.z), 4 * g + 2);
    f(__uint_as_float(x.w), 4 * g + 3);
  } else {
    f(half_word<GD>(x.x & 0xffffu), 8 * g);
    f(half_word<GD>(x.x >> 16), 8 * g + 1);
    f(half_word<GD>(x.y & 0xffffu), 8 * g + 2);
    f(half_word<GD>(x.y >> 16), 8 * g + 3);
    f(half_word<GD>(x.z & 0xffffu), 8 * g + 4);
    f(half_word<GD>(x.z >> 16), 8 * g + 5);
    f(half_word<GD>(x.w & 0xffffu), 8 * g + 6);
    f(half_word<GD>(x.w >> 16), 8 * g + 7);
  }
}

// Calls f(x, j) for j = 0 .. E-1 in order and returns f (the functor carries its state by value, so that it
// stays in registers).  16-byte granules (4 fp32 or 8 half values) when the row allows.
template <int GD, typename F>
__device__ __forceinline__ F walk_row(const void* row, int E, F f) {
  constexpr int V = GD == LANCET_F32 ? 4 : 8;
  const bool vec = ((E & (V - 1)) == 0) && ((reinterpret_cast<uintptr_t>(row) & 15u) == 0);
  if (vec) {
    const u32x4* r = static_cast<const u32x4*>(row);
    const int n = E / V;
    // Rows longer than a line: eight granules (one 128-byte line) are loaded before any of them is used (5-10 %
    // on routing with hundreds of experts).  The last block of up to eight granules, which is all of a short row,
    // is walked load by load (measured faster for rows of one line and less).
    constexpr int kAhead = 8;
    for (int g0 = 0; g0 < n - kAhead; g0 += kAhead) {
      u32x4 xs[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) xs[i] = r[g0 + i];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) walk_granule<GD>(xs[i], g0 + i, f);
    }
    for (int g = n > kAhead ? (n - 1) / kAhead * kAhead : 0; g < n; ++g) walk_granule<GD>(r[g], g, f);
  } else {
    for (int j = 0; j < E; ++j) f(gate_at<GD>(row, j), j);
  }
  return f;
}

template <int K>
struct SelectTop {
  TopState t;
  __device__ __forceinline__ void operator()(float x, int j) { t = consider<K>(t, x, j); }
};
// Selection and the softmax denominator in one walk: the sum is kept relative to the running maximum and
// rescaled when a larger value comes (the values the two-pass form adds, exp(x - max), each within an ulp or two;
// used where the row is staged through LDS and a second walk would move it through LDS again).
template <int K>
struct SelectSum {
  TopState t;
  float sum;
  __device__ __forceinline__ void operator()(float x, int j) {
    const bool first = (t.i1 < 0) | (x > t.v1);
    if (first) sum = (t.i1 < 0 ? 0.f : sum * __expf(t.v1 - x)) + 1.f;
    else sum += __expf(x - t.v1);
    t = consider<K>(t, x, j);
  }
};
// The terms of the denominator go through the hardware exponential (__expf); the two gate values themselves
// through expf.  Against an fp64 softmax the gates are as close as with expf in the sum (largest relative error
// 4e-7 at 32 experts, 1.6e-6 at 512, either way: what shows is the rounding of the fp32 sum), and routing with
// 64 experts or more takes 10-15 % less time.
struct SumExp {  // sequential sum in expert order
  float top, sum;
  __device__ __forceinline__ void operator()(float x, int) { sum += __expf(x - top); }
};

// noise (K = 2 only, may be null): values added to the row for the second choice alone, the first
// choice masked out (docker/resources/sharded_moe.py:275-278); gate values always come from the row.
// Row and noise are stored as GD; 16-bit values tie massively, and the first maximum wins as always.
template <int K, int GD>
__device__ __forceinline__ Routed route_token(const void* __restrict__ row, const void* __restrict__ noise, int E,
                                              bool is_logits) {
  SelectTop<K> sel = {{0.f, 0.f, -1, -1}};
  TopState t = walk_row<GD>(row, E, sel).t;
  if (K == 2 && noise) {
    // second choice again, on row + noise: first max over the experts other than the first choice
    float best = 0.f;
    t.i2 = -1;
    for (int j = 0; j < E; ++j) {
      const float x = gate_at<GD>(row, j);
      const float y = x + gate_at<GD>(noise, j);
      const bool take = (j != t.i1) & ((t.i2 < 0) | (y > best));
      best = take ? y : best;
      t.v2 = take ? x : t.v2;
      t.i2 = take ? j : t.i2;
    }
  }
  float sum = 1.f;
  if (is_logits) {
    SumExp se = {t.v1, 0.f};
    sum = walk_row<GD>(row, E, se).sum;
  }
  Routed r;
  r.e0 = t.i1;
  r.p0 = is_logits ? expf(t.v1 - t.v1) / sum : t.v1;
  r.e1 = K == 2 ? t.i2 : -1;
  r.p1 = K == 2 ? (is_logits ? expf(t.v2 - t.v1) / sum : t.v2) : 0.f;
  return r;
}

// ---- rows held in registers ---------------------------------------------------------------------------------
// A row of up to kHeldGranules 16-byte granules is taken by 2^q neighbouring lanes, four granules each, all loads in
// flight together and the next rows' behind them; what the lanes chose is merged by shuffles, and the exponentials are
// summed from the registers once the row's maximum is known.  The kernel is bound by its vector instructions (262144
// tokens x 64 fp32 experts: 67 MB, which memory delivers in 11 us), so nothing is decided per element that can be decided
// per row: the running choice starts from "none" at -inf, and the rows that this does not describe (a NaN, a row whose
// choice is -inf, an infinite sum) are told by their outcome and walked again one by one by route_token.
// First routing kernel, before (rows walked by one lane each, through LDS where they are longer than a line, element by
// element where they are not whole granules) and after, us: 262144 x 64 fp32 top-1 27.0 -> 17.7, 65536 x 32 fp32 top-2
// 9.6 -> 8.5, 10007 x 60 bf16 top-2 21 -> 8.3.  The sum is formed from 16 terms (32 of 16 bits) per lane and then over the
// lanes: largest relative error of a gate value at 64 / 256 experts 6.4e-7 / 1.2e-6 before, 3.6e-7 / 2.3e-7 after.
constexpr int kHeldPerLane = 4;
constexpr int kHeldGranules = 16 * kHeldPerLane;
typedef u32x4 u32x4_gate __attribute__((aligned(2)));

// Which rows are held (`gate` values of gb bytes, no noise).  Rows of 3 to 64 granules that are not whole granules or not
// aligned to them: all, whatever the batch (the walk takes them value by value: 2048 x 31 fp32 13.6 us, held 7.5).  Aligned
// rows of whole granules, where the walk is a load per granule (walked / held, top-1, us):
//   * the lanes of a row take n = 4, 8, 16, 32 or 64 granules and do the work of all whether the row has them or not, so
//     that a row of 36 costs as much as one of 64: 16384 x 144 fp32 logits 18.0 / 25.6, x 256 22.6 / 22.7.  In short launches
//     only full lanes pay, and rows of up to 16 granules of which one in eight is missing (2048 x 60 fp32 9.9 / 9.5, x 52
//     9.2 / 9.5; in less than a tile a tenth slower).  From 384 tiles on, where the walk's lines no longer survive in the cache
//     from one load to the next, three quarters are enough (98304 x 96 fp32 27.7 / 23.6, 65536 of them 30.1 / 30.2), and
//     from 512 tiles on any row of more than the line that a walk reads at once (131072 x 144 fp32 42.9 / 35.9);
//   * fp32 rows of more than 16 granules in less than a tile: a wave has 16 and more rounds of them to itself, one after
//     the other, where the walk has one (64 x 256 logits 13.4 / 16.1);
//   * without the softmax the walk is a few compares per value, and only the cache decides: from 512 tiles and a whole line
//     on (131072 x 64 fp32 19.1 / 15.0; 98304 x 128 18.9 / 21.0).
// The choice is the same either way.
constexpr int kStageMinTiles = 512;
constexpr int kHeldPackedTiles = 384;
inline bool rows_are_held(const void* gate, const void* noise, int S, int E, int gb, bool is_logits) {
  const int bytes = E * gb, n = bytes / 16;
  if (noise != nullptr || bytes <= 32 || bytes > 16 * kHeldGranules) return false;
  if (bytes % 16 != 0 || (reinterpret_cast<uintptr_t>(gate) & 15u) != 0) return true;
  const int tiles = (S + kTile - 1) / kTile;
  int taken = kHeldPerLane;
  while (taken < n) taken *= 2;
  const bool packed = 4 * n >= 3 * taken;
  if (!is_logits) return tiles >= kStageMinTiles && n >= 8 && packed;
  if (tiles >= kStageMinTiles) return n > 8 || packed;
  if (tiles >= kHeldPackedTiles) return packed;
  if (n < taken) return n <= 16 && 8 * n >= 7 * taken && tiles >= 4;
  return n <= 16 || gb == 2 || S >= kTile;
}

// f(x, i) for the values of a granule as fp32; i is the value's place in it
template <int GD, typename F>
__device__ __forceinline__ void each_value(const u32x4& x, F f) {
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (GD == LANCET_F32) {
      f(__uint_as_float(x[w]), w);
    } else {
      f(half_word<GD>(x[w] & 0xffffu), 2 * w);
      f(half_word<GD>(x[w] >> 16), 2 * w + 1);
    }
  }
}

constexpr int kNoExpert = 0x7fffffff;

// The value of the partner in merge step 0 .. 3 of a group of up to 16 lanes that agree inside their half of it: the
// neighbour, the pair's, the quad's and the half row's mirror image.  (Register moves: a shuffle goes through LDS, and the
// merges of a round are a serial chain; selection of 32768 x 64 8.0 -> 7.5 us.)
template <int STEP>
__device__ __forceinline__ int merge_partner(int x) {
  constexpr int ctrl = STEP == 0 ? 0xb1 : STEP == 1 ? 0x4e : STEP == 2 ? 0x141 : 0x140;
  return __builtin_amdgcn_update_dpp(0, x, ctrl, 0xf, 0xf, false);
}
template <int STEP>
__device__ __forceinline__ float merge_partner(float x) {
  return __int_as_float(merge_partner<STEP>(__float_as_int(x)));
}
// f(step) for the merge steps of a group of 2^q lanes
template <typename F>
__device__ __forceinline__ void merge_steps(int q, F f) {
  if (q > 0) f(std::integral_constant<int, 0>());
  if (q > 1) f(std::integral_constant<int, 1>());
  if (q > 2) f(std::integral_constant<int, 2>());
  if (q > 3) f(std::integral_constant<int, 3>());
}

// what route_token returns, for the lane's token of the wave's nrows <= 64 consecutive ones from `rows` on (lanes past
// them: anything).  All lanes of the wave, uniform control flow.
// WIDE: a lane takes one, two or four granules, so many lanes to a row that the wave's 16 rows fill it.
template <int K, int GD, bool WIDE = false>
__device__ __forceinline__ Routed route_rows_held(const char* rows, int nrows, int E, bool is_logits) {
  constexpr int gb = GD == LANCET_F32 ? 4 : 2;
  constexpr int V = 16 / gb;
  const int lane = lane_id();
  const uint32_t row_bytes = static_cast<uint32_t>(E) * gb;
  const int n = static_cast<int>((row_bytes + 15u) / 16u);
  const int mine_n = !WIDE || n > 8 ? kHeldPerLane : n > 4 ? 2 : 1;  // granules per lane
  int q = 0;
  while (mine_n << q < n) ++q;
  const int width = 1 << q, per_round = kWave >> q;  // lanes per row, rows per round
  const int sub = lane & (width - 1);
  // where the lane's granules lie in a row; the last of a row that is not whole granules is drawn back to end with it, and
  // the values it shares with the one before (the first `dup`) count as -inf
  uint32_t at[kHeldPerLane];
  int dup[kHeldPerLane];
#pragma unroll
  for (int k = 0; k < kHeldPerLane; ++k) {
    const int g = k * width + sub;
    at[k] = min(16u * static_cast<uint32_t>(g), row_bytes - 16u);
    dup[k] = g < n ? static_cast<int>(16u * static_cast<uint32_t>(g) - at[k]) / gb : V;
  }
  const bool ragged = n * 16 != static_cast<int>(row_bytes) || n != mine_n * width;
  const auto load = [&](int r, u32x4 (&x)[kHeldPerLane]) {
    const int row = r * per_round + (lane >> q);
    const char* p = rows + static_cast<size_t>(min(row, nrows - 1)) * row_bytes;
#pragma unroll
    for (int k = 0; k < kHeldPerLane; ++k)
      if (!WIDE || k < mine_n) x[k] = *reinterpret_cast<const u32x4_gate*>(p + at[k]);
  };
  const int rounds = (nrows + per_round - 1) / per_round;
  float v1 = 0.f, v2 = 0.f, sum = 0.f;  // the lane's own token
  int i1 = 0, i2 = 0;
  u32x4 x[kHeldPerLane], nx[kHeldPerLane];
  if (!WIDE) load(0, x);
  for (int r = 0; r < rounds; ++r) {
    if (WIDE) load(r, x);  // sixteen waves: another one's loads are on their way
    else if (r + 1 < rounds) load(r + 1, nx);
    float f[kHeldPerLane][V];
#pragma unroll
    for (int k = 0; k < kHeldPerLane; ++k) each_value<GD>(x[k], [&](float val, int i) { f[k][i] = val; });
    if (ragged) {
#pragma unroll
      for (int k = 0; k < kHeldPerLane; ++k)
#pragma unroll
        for (int i = 0; i < V; ++i) f[k][i] = i < dup[k] ? -INFINITY : f[k][i];
    }
    float a1 = -INFINITY, a2 = -INFINITY;
    int j1 = kNoExpert, j2 = kNoExpert;
#pragma unroll
    for (int k = 0; k < kHeldPerLane; ++k) {
      if (WIDE && k >= mine_n) break;
      const int j0 = static_cast<int>(at[k] / gb);
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const float val = f[k][i];
        const bool first = val > a1;
        if (K == 2) {
          const bool second = val > a2;
          a2 = first ? a1 : (second ? val : a2);
          j2 = first ? j1 : (second ? j0 + i : j2);
        }
        a1 = first ? val : a1;
        j1 = first ? j0 + i : j1;
      }
    }
    merge_steps(q, [&](auto step) {
      const float b1 = merge_partner<step.value>(a1);
      const int k1 = merge_partner<step.value>(j1);
      const bool theirs = (b1 > a1) | ((b1 == a1) & (k1 < j1));  // equal values: the first expert
      if (K == 2) {
        const float b2 = merge_partner<step.value>(a2);
        const int k2 = merge_partner<step.value>(j2);
        // the second choice is the loser of the two firsts or the winner's own second
        const float c = theirs ? a1 : b1, d = theirs ? b2 : a2;
        const int cj = theirs ? j1 : k1, dj = theirs ? k2 : j2;
        const bool loser = (c > d) | ((c == d) & (cj < dj));
        a2 = loser ? c : d;
        j2 = loser ? cj : dj;
      }
      a1 = theirs ? b1 : a1;
      j1 = theirs ? k1 : j1;
    });
    float part = 0.f;
#pragma unroll
    for (int k = 0; k < kHeldPerLane; ++k) {
      if (WIDE && k >= mine_n) break;
#pragma unroll
      for (int i = 0; i < V; ++i) part += is_logits ? __expf(f[k][i] - a1) : f[k][i];
    }
    merge_steps(q, [&](auto step) { part += merge_partner<step.value>(part); });
    // the round's tokens to their lanes
    const int from = (lane & (per_round - 1)) << q;
    const bool mine = lane / per_round == r;
    const float t1 = __shfl(a1, from, kWave), ts = __shfl(part, from, kWave);
    const int u1 = __shfl(j1, from, kWave);
    v1 = mine ? t1 : v1;
    i1 = mine ? u1 : i1;
    sum = mine ? ts : sum;
    if (K == 2) {
      const float t2 = __shfl(a2, from, kWave);
      const int u2 = __shfl(j2, from, kWave);
      v2 = mine ? t2 : v2;
      i2 = mine ? u2 : i2;
    }
#pragma unroll
    for (int k = 0; k < kHeldPerLane && !WIDE; ++k) x[k] = nx[k];
  }
  Routed res;
  const bool plain = sum == sum && i1 != kNoExpert && (K == 1 || i2 != kNoExpert);
  if (plain || lane >= nrows) {
    res.e0 = i1;
    res.p0 = is_logits ? 1.f / sum : v1;
    res.e1 = K == 2 ? i2 : -1;
    res.p1 = K == 2 ? (is_logits ? expf(v2 - v1) / sum : v2) : 0.f;
  } else {
    res = route_token<K, GD>(rows + static_cast<size_t>(lane) * row_bytes, nullptr, E, is_logits);
  }
  return res;
}

// ---- rows longer than a cache line: staged through LDS ------------------------------------------------------
// A lane that walks its own row touches each 128-byte line of it in eight loads, and every load of the wave
// touches 64 different lines; with rows of several lines and many waves on a CU the lines are evicted between a
// lane's visits and fetched again.  Such rows, where they are not held in registers, are therefore read the way they lie in
// memory, a wave's 64 rows 128 bytes at a time (eight lanes per row and line, every line whole in one load), passed through
// LDS and walked from there, each lane its own row as before: the values and their order are the same, so is the result.  It
// pays from about two workgroups per CU on (kStageMinTiles: 262144 rows of 256 fp32 experts 274 -> 92 us); launches of fewer
// tiles keep the direct walk, whose lines survive in the cache (65536 of them, top-2, 50 against 64).
constexpr int kStageChunk = 128;                   // bytes of a row staged at a time
constexpr int kStageRow = kStageChunk + 16;        // row pitch in LDS (the pad spreads the lanes' reads over the banks)
constexpr int kStageWave = kWave * kStageRow;      // bytes per wave
constexpr int kStageBytes = kWavesPerTile * kStageWave;

template <int GD>
__host__ __device__ inline bool rows_are_staged(const void* gate, const void* noise, int S, int E) {
  constexpr int gb = GD == LANCET_F32 ? 4 : 2;
  return noise == nullptr && (S + kTile - 1) / kTile >= kStageMinTiles && E * gb > kStageChunk && (E * gb) % 16 == 0 &&
         (reinterpret_cast<uintptr_t>(gate) & 15u) == 0;
}

// Calls f(x, j), j = 0 .. E-1 in order, for the lane's row of the wave's rows (rows = first of them, nrows <= 64
// valid ones, E * sizeof(value) a multiple of 16, 16-byte aligned).  All lanes of the wave, uniform control flow;
// stage = the wave's kStageWave bytes of LDS.
// the lane's eight granules of chunk c0 of the wave's rows (zeros beyond the rows and beyond the chunk)
__device__ __forceinline__ void stage_load(const char* rows, int nrows, int row_bytes, int c0, u32x4 (&x)[8]) {
  const int lane = lane_id();
  const int gpr = min(kStageChunk, row_bytes - c0) / 16;  // granules per row in this chunk: 8, less in the last
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int g = i * kWave + lane;
    const int r = gpr == 8 ? (g >> 3) : g / gpr;
    const int part = gpr == 8 ? (g & 7) : g - r * gpr;
    x[i] = u32x4{0u, 0u, 0u, 0u};
    if (r < nrows) x[i] = *reinterpret_cast<const u32x4*>(rows + static_cast<size_t>(r) * row_bytes + c0 + part * 16);
  }
}

template <int GD, typename F>
__device__ __forceinline__ F walk_rows_staged(const char* rows, int nrows, int E, char* stage, F f) {
  constexpr int gb = GD == LANCET_F32 ? 4 : 2;
  constexpr int V = 16 / gb;  // values per 16-byte granule
  const int row_bytes = E * gb;
  const int lane = lane_id();
  u32x4 x[8], nx[8];
  stage_load(rows, nrows, row_bytes, 0, x);
  for (int c0 = 0; c0 < row_bytes; c0 += kStageChunk) {
    const int gpr = min(kStageChunk, row_bytes - c0) / 16;
    // the next chunk's loads are in flight while this one is walked
    const bool more = c0 + kStageChunk < row_bytes;
    if (more) stage_load(rows, nrows, row_bytes, c0 + kStageChunk, nx);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int g = i * kWave + lane;
      const int r = gpr == 8 ? (g >> 3) : g / gpr;
      const int part = gpr == 8 ? (g & 7) : g - r * gpr;
      if (r < kWave) *reinterpret_cast<u32x4*>(stage + r * kStageRow + part * 16) = x[i];
    }
    // the wave's own LDS traffic is in order; the fences keep the compiler from moving the reads above the writes
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int j0 = c0 / gb;
    for (int p = 0; p < gpr; ++p) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(stage + lane * kStageRow + p * 16);
      const int j = j0 + p * V;
      if (GD == LANCET_F32) {
        f(__uint_as_float(v.x), j);
        f(__uint_as_float(v.y), j + 1);
        f(__uint_as_float(v.z), j + 2);
        f(__uint_as_float(v.w), j + 3);
      } else {
        f(half_word<GD>(v.x & 0xffffu), j);
        f(half_word<GD>(v.x >> 16), j + 1);
        f(half_word<GD>(v.y & 0xffffu), j + 2);
        f(half_word<GD>(v.y >> 16), j + 3);
        f(half_word<GD>(v.z & 0xffffu), j + 4);
        f(half_word<GD>(v.z >> 16), j + 5);
        f(half_word<GD>(v.w & 0xffffu), j + 6);
        f(half_word<GD>(v.w >> 16), j + 7);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (more) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = nx[i];
    }
  }
  return f;
}

// ---- how a kernel selects ------------------------------------------------------------------------------------------
enum SelectForm { kWalkRows = 0, kHoldRows = 1, kHoldWide = 2 };
// Threads of a workgroup that selects for a tile.  Wide: sixteen waves select sixteen tokens each and hand what they chose to the
// four that go on.  A short launch is over when its waves are, and a wave's 64 rows of a few granules were four rounds of
// loads, compares and exponentials one after the other.
template <int FORM>
constexpr int kSelectThreadsOf = FORM == kHoldWide ? 4 * kTile : kTile;
constexpr int kWideRows = kTile / 16;

// Selection for token s of a workgroup whose thread t < kTile holds token s = first + t (kTile consecutive tokens): what
// route_token gives, from registers (kHoldRows, kHoldWide: select_launch), by the direct walk or through LDS.  All threads,
// uniform control flow; lds = at least kStageBytes when rows_are_staged (it may be reused after the
// call).  Threads with s >= S get {-1, -1, 0, 0}.  kHoldWide: threads from kTile on have nothing left to do.
template <int K, int GD, int FORM>
__device__ __forceinline__ Routed route_tile_token(const void* gate, const void* noise, int s, int S, int E, bool is_logits,
                                                   void* lds) {
  constexpr size_t gb = GD == LANCET_F32 ? 4 : 2;
  Routed r = {-1, -1, 0.f, 0.f};
  if constexpr (FORM == kHoldWide) {
    __shared__ Routed chosen[kTile];
    const int w = static_cast<int>(threadIdx.x) / kWave, lane = lane_id();
    const int first = s - static_cast<int>(threadIdx.x) + w * kWideRows;
    const int nrows = min(S - first, kWideRows);
    if (nrows > 0) {
      const Routed held = route_rows_held<K, GD, true>(static_cast<const char*>(gate) + static_cast<size_t>(first) * E * gb, nrows, E, is_logits);
      if (lane < nrows) chosen[w * kWideRows + lane] = held;
    }
    __syncthreads();
    if (threadIdx.x < kTile && s < S) r = chosen[threadIdx.x];
    return r;
  }
  if constexpr (FORM == kHoldRows) {
    const int first = s - lane_id();  // the wave's first token
    if (first < S) {
      const Routed held = route_rows_held<K, GD>(static_cast<const char*>(gate) + static_cast<size_t>(first) * E * gb,
                                                 min(S - first, kWave), E, is_logits);
      if (s < S) r = held;
    }
    return r;
  }
  if (!rows_are_staged<GD>(gate, noise, S, E)) {
    if (s < S) {
      const size_t off = static_cast<size_t>(s) * E * gb;
      r = route_token<K, GD>(static_cast<const char*>(gate) + off, noise ? static_cast<const char*>(noise) + off : nullptr, E,
                             is_logits);
    }
    return r;
  }
  const int first = s - lane_id();  // the wave's first token
  const int nrows = min(max(S - first, 0), kWave);
  const char* rows = static_cast<const char*>(gate) + static_cast<size_t>(first) * E * gb;
  char* stage = static_cast<char*>(lds) + (threadIdx.x / kWave) * kStageWave;
  TopState t;
  float sum = 1.f;
  if (is_logits) {
    SelectSum<K> sel = {{0.f, 0.f, -1, -1}, 0.f};
    sel = walk_rows_staged<GD>(rows, nrows, E, stage, sel);
    t = sel.t;
    sum = sel.sum;
  } else {
    SelectTop<K> sel = {{0.f, 0.f, -1, -1}};
    t = walk_rows_staged<GD>(rows, nrows, E, stage, sel).t;
  }
  if (s < S) {
    r.e0 = t.i1;
    r.p0 = is_logits ? expf(t.v1 - t.v1) / sum : t.v1;
    r.e1 = K == 2 ? t.i2 : -1;
    r.p1 = K == 2 ? (is_logits ? expf(t.v2 - t.v1) / sum : t.v2) : 0.f;
  }
  __syncthreads();  // the caller may use the LDS for something else now
  return r;
}

// GD as a compile-time constant inside `...` for the run-time code gd
#define LANCET_GATE_SWITCH(gd, ...)                                \
  switch (gd) {                                                    \
    case LANCET_BF16: { constexpr int GD = LANCET_BF16; __VA_ARGS__; } break; \
    case LANCET_F16: { constexpr int GD = LANCET_F16; __VA_ARGS__; } break;   \
    default: { constexpr int GD = LANCET_F32; __VA_ARGS__; } break;           \
  }

// GD and FORM as compile-time constants inside `...`
#define LANCET_SELECT_SWITCH(gd, form, ...)                                                              \
  LANCET_GATE_SWITCH(gd, if (form == kHoldWide) { constexpr int FORM = kHoldWide; __VA_ARGS__; }           \
                         else if (form == kHoldRows) { constexpr int FORM = kHoldRows; __VA_ARGS__; }      \
                         else { constexpr int FORM = kWalkRows; __VA_ARGS__; })

// how a kernel that selects is launched: its form, its threads and the LDS its selection needs
struct SelectLaunch {
  SelectForm form;
  int threads;
  size_t lds;
};
// Wide: short launches (a tile has a CU to itself) of rows long enough for the second barrier and the waves that are started to
// pay, where few lanes take granules that the row has not (as in rows_are_held).  moe_encode of 256 / 4096 / 65536 tokens,
// otherwise / wide, us: 64 fp32 logits top-1 7.3 / 5.6, 10.5 / 8.9, 16.7 / 14.9, top-2 8.8 / 7.7, 12.5 / 11.4, 23.9 / 22.5; 128 top-1
// 11.2 / 7.3, 14.6 / 10.6, 24.1 / 20.8; 256 21.8 / 13.1, 22.7 / 14.0, 34.5 / 30.3; but 32 top-2 6.5 / 6.9, 9.9 / 10.2 and 16 6.1 / 7.2.  128
// bf16 logits top-2 11.3 / 10.6, 15.2 / 14.1, 64 8.1 / 8.6.  131072 tokens: 64 fp32 23.8 / 24.8.  The rest is moe_route alone:
//   * logits of more than half a tile: five lanes in eight, whatever the type.  256 tokens top-2: 68 fp32 (17 granules, lanes for
//     32) 10.0 / 11.1, 76 10.9 / 11.2, 80 11.2 / 11.2, 96 13.8 / 11.4; 132 (33 of 64) 13.2 / 16.4, 152 15.4 / 16.4, 160 18.8 / 16.4; 136 bf16
//     14.3 / 16.0, 160 15.8 / 15.9, 272 22.1 / 25.1, 320 26.5 / 25.3; 4096 tokens top-1: 132 fp32 12.3 / 14.2, 144 14.5 / 15.2, 160 18.4 / 15.3,
//     272 bf16 19.5 / 22.0, 320 23.5 / 22.0.  Rows that are not whole aligned granules are held otherwise, by the same lanes, and
//     always gain (65 fp32 14.3 / 11.1, 129 23.6 / 16.4, 257 bf16 31.9 / 24.9), and so do few tokens (64: 132 fp32 12.8 / 11.3; moe_encode of
//     128: 72 fp32 8.6 / 7.9, 136 bf16 16.4 / 14.3);
//   * probabilities, which are a few compares per value: all lanes, four granules each.  256 tokens top-1: 64 fp32 6.8 / 6.3, 128
//     8.6 / 7.8, 256 12.1 / 10.8, 128 bf16 8.4 / 7.9, 256 11.5 / 10.2, 512 17.9 / 15.8; 65536 top-2: 64 fp32 15.2 / 14.2, 128 bf16 19.9 / 18.2, 512
//     46.0 / 40.4; but lanes with two granules and fewer 32 fp32 5.6 / 5.9, 64 bf16 6.1 / 6.8, and lanes without, 120 fp32 7.2 / 7.6, 200
//     9.0 / 11.1.  What fills the lanes and is not whole granules gains too (1000 tokens: 61 fp32 9.2 / 8.3, 253 20.2 / 13.3, 505 bf16
//     27.6 / 20.3), but for the tokens of one of the sixteen waves (16: 253 fp32 7.2 / 7.4).  64 granules of fp32: the walk is faster
//     again from 193 tiles on (49152 tokens 21.6 / 20.8, 65536 22.9 / 25.9).
constexpr int kWideTiles = 256;
constexpr int kWideLongTiles = 192;
inline bool rows_are_wide(const void* gate, const void* noise, int S, int E, int gb, bool is_logits) {
  const int bytes = E * gb, n = (bytes + 15) / 16, tiles = (S + kTile - 1) / kTile;
  if (noise != nullptr || bytes <= 32 || bytes > 16 * kHeldGranules || tiles > kWideTiles) return false;
  int taken = kHeldPerLane;
  while (taken < n) taken *= 2;
  const bool walked = bytes % 16 == 0 && (reinterpret_cast<uintptr_t>(gate) & 15u) == 0;  // otherwise held
  if (!is_logits) {
    if (n != taken || n <= 8 || (!walked && S <= kWideRows)) return false;
    return !walked || gb == 2 || n < kHeldGranules || tiles <= kWideLongTiles;
  }
  return E >= (S <= kWave ? 32 : gb == 4 ? 56 : 96) && (!walked || S <= kTile / 2 || 8 * n >= 5 * taken);
}
inline SelectLaunch select_launch(int gate_dtype, const void* gate, const void* noise, int S, int E, bool is_logits) {
  const int gb = gate_dtype == LANCET_F32 ? 4 : 2;
  if (rows_are_wide(gate, noise, S, E, gb, is_logits)) return {kHoldWide, kSelectThreadsOf<kHoldWide>, 0};
  if (rows_are_held(gate, noise, S, E, gb, is_logits)) return {kHoldRows, kTile, 0};
  SelectLaunch l = {kWalkRows, kTile, 0};
  LANCET_GATE_SWITCH(gate_dtype, l.lds = rows_are_staged<GD>(gate, noise, S, E) ? kStageBytes : 0)
  return l;
}

}  // namespace lancet
