// moe_encode of few tokens: routing and row movement in one launch (a tile of tokens) or two (a few tiles) instead of two to
// four.  What bounds such a call is its chain of launches: each of the kernels it replaces takes 2.5 to 8 us, the length of a
// kernel that starts, makes two or three dependent memory round trips and ends, and the next one starts 1 us later.
#include "launchers.hpp"
#include "route.hpp"
#include <algorithm>

namespace lancet {


struct EncodeArgs {
  RouteArgs r;
  const char* data;
  char* out;
  uint32_t row_bytes;
  int q;              // 2^q lanes of a workgroup share one token row
  int tokens;         // tokens per workgroup: a power of two, kTile at most
  int token_blocks;
  int tail_rows;      // rows that a tail workgroup clears in a turn
  int tail_chunks;    // turns that clear an expert's rows if none is used (0: nobody clears them)
  int tail_blocks;    // workgroups that clear: one tile: of all experts; a few tiles: of each expert
  int rows_at_used;   // rows start behind those that earlier calls used
  int needs_setup;    // the outputs are marked where the workspace was never set up
};

typedef u32x4 u32x4_any __attribute__((aligned(2)));

// A row is moved in 16-byte granules at any alignment, the last one drawn back to end with it (its first bytes are written
// twice, with the same values); rows of less than a granule two bytes at a time.  Non-temporal both ways: 6000 x 1024 top-1
// 10.8 us against 12.5 with plain accesses, 6000 x 1003 11.4 against 13.2.
struct RowCopy {
  uint32_t row_bytes;
  int units;
  __device__ __forceinline__ explicit RowCopy(uint32_t bytes)
      : row_bytes(bytes), units(static_cast<int>(bytes >= 16u ? (bytes - 1u) / 16u + 1u : bytes / 2u)) {}
  __device__ __forceinline__ u32x4 load(const char* row, int v) const {
    if (row_bytes >= 16u) return __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(row + at(v)));
    u32x4 x = {0u, 0u, 0u, 0u};
    x.x = *reinterpret_cast<const uint16_t*>(row + 2 * v);
    return x;
  }
  __device__ __forceinline__ void store(LANCET_GLOBAL char* row, int v, u32x4 x) const {
    if (row_bytes >= 16u) __builtin_nontemporal_store(x, (LANCET_GLOBAL u32x4_any*)(row + at(v)));
    else *(LANCET_GLOBAL uint16_t*)(row + 2 * v) = static_cast<uint16_t>(x.x);
  }
  __device__ __forceinline__ uint32_t at(int v) const { return min(16u * static_cast<uint32_t>(v), row_bytes - 16u); }
};

// The workgroup's rows: thread tid starts with granules v, v + step of row r, asked for before the routing is known.
struct RowWork {
  int r, v, step, per_round;
  u32x4 x0, x1;
  __device__ __forceinline__ void load(const EncodeArgs& a, const RowCopy& c, int first, int n) {
    x0 = x1 = u32x4{0u, 0u, 0u, 0u};
    const char* row = a.data + static_cast<size_t>(first + r) * a.row_bytes;
    if (r < n && v < c.units) x0 = c.load(row, v);
    if (r < n && v + step < c.units) x1 = c.load(row, v + step);
  }
  __device__ __forceinline__ RowWork(const EncodeArgs& a, const RowCopy& c, int first, int n) {
    step = 1 << a.q, per_round = kTile >> a.q;
    r = static_cast<int>(threadIdx.x) >> a.q, v = static_cast<int>(threadIdx.x) & (step - 1);
    load(a, c, first, n);
  }
  // s_dest[j * kTile + i]: row of the buffer that slot j of the workgroup's token i goes to, or -1
  template <int K>
  __device__ __forceinline__ void store(const EncodeArgs& a, const RowCopy& c, int first, int n, const int* s_dest) {
    while (r < n) {
      const int row = r;
      u32x4 y0 = x0, y1 = x1;
      r += per_round;
      load(a, c, first, n);  // the next row's granules are on their way while this one's are written
      LANCET_GLOBAL char* dst[K];
      bool any = false;
#pragma unroll
      for (int j = 0; j < K; ++j) {
        const int d = s_dest[j * kTile + row];
        dst[j] = d < 0 ? nullptr : as_global(a.out + static_cast<size_t>(d) * a.row_bytes);
        any = any || d >= 0;
      }
      if (!any) continue;
      const char* src = a.data + static_cast<size_t>(first + row) * a.row_bytes;
      for (int u = v;;) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
          if (!dst[j]) continue;
          if (u < c.units) c.store(dst[j], u, y0);
          if (u + step < c.units) c.store(dst[j], u + step, y1);
        }
        u += 2 * step;
        if (u >= c.units) break;
        y0 = c.load(src, u);
        if (u + step < c.units) y1 = c.load(src, u + step);
      }
    }
  }
};

__device__ __forceinline__ int buffer_row(const EncodeArgs& a, int e, int l) {
  if (e < 0 || l < 0) return -1;
  if (a.rows_at_used && a.r.used_in) l += a.r.used_in[e];
  return l < a.r.C ? e * a.r.C + l : -1;
}

// the first of an expert's rows that is to be cleared; total = tokens of the batch that chose it (rows of earlier calls are in
// the buffer already where this call's start behind them)
__device__ __forceinline__ int64_t tail_start(const EncodeArgs& a, int e, int64_t total, bool marked) {
  const int64_t used_in = a.r.used_in ? a.r.used_in[e] : 0;
  const int64_t used_out = min(used_in + total, static_cast<int64_t>(a.r.C));
  return marked ? 0 : max(used_out - (a.rows_at_used ? 0 : used_in), static_cast<int64_t>(0));
}
// a turn: tail_rows rows of the expert's tail, which starts at row `from`
__device__ __forceinline__ void clear_tail(const EncodeArgs& a, int e, int64_t from, int chunk) {
  const int64_t first = from + static_cast<int64_t>(chunk) * a.tail_rows;
  const int64_t last = min(first + a.tail_rows, static_cast<int64_t>(a.r.C));
  if (first >= last) return;
  LANCET_GLOBAL char* run = as_global(a.out + (static_cast<size_t>(e) * a.r.C + first) * a.row_bytes);
  const size_t bytes = static_cast<size_t>(last - first) * a.row_bytes;
  const u32x4 z = {0u, 0u, 0u, 0u};
  if (bytes >= 16) {
    for (size_t v = threadIdx.x; 16 * v < bytes; v += kTile) *(LANCET_GLOBAL u32x4_any*)(run + min(16 * v, bytes - 16)) = z;
  } else {
    for (size_t v = threadIdx.x; 2 * v < bytes; v += kTile) *(LANCET_GLOBAL uint16_t*)(run + 2 * v) = 0;
  }
}

// used capacity and element counts of all experts; totals[c] = tokens of counter c
template <int K>
__device__ __forceinline__ void store_totals(const RouteArgs& r, const uint32_t* totals, bool marked) {
  for (int c = threadIdx.x; c < r.E; c += kTile) {
    const int64_t used = r.used_in ? r.used_in[c] : 0;
    const int64_t total = static_cast<int64_t>(totals[c]) + (K == 2 ? totals[r.E + c] : 0u);
    const int64_t uo = min(used + total, static_cast<int64_t>(r.C));
    r.used_out[c] = marked ? -1 : static_cast<int32_t>(uo);
    r.elems_out[c] = marked ? 0 : static_cast<uint64_t>((uo - used) * r.M);
  }
}

// the look-back form's contract: memory that was never set up yields marks, and says so
__device__ __forceinline__ bool not_set_up(const EncodeArgs& a) {
  if (!a.needs_setup || ld_agent(a.r.ws.hdr + kWsMagic) == kWsMagicValue) return false;
  if (blockIdx.x == 0 && threadIdx.x == 0) st_agent(a.r.ws.hdr + kWsError, 1u);
  return true;
}

// A tile of tokens (256 and less): every workgroup routes all of them, a token per thread, and moves its own rows; the first
// also writes the routing.  Routing 64 tokens x 8 experts again in each of 48 workgroups costs nothing that is not waited for
// anyway: 64 x 1024 bf16 top-2, 8 experts, 9.1 us as three kernels (count, place, scatter), 4.6 as this one.
template <int K, int GD, int FORM>
__global__ __launch_bounds__(kSelectThreadsOf<FORM>) void encode_tile_kernel(EncodeArgs a) {
  extern __shared__ uint32_t s_cnt[];
  __shared__ int s_dest[K * kTile];
  const RouteArgs& r = a.r;
  const int tid = threadIdx.x;
  const bool mover = static_cast<int>(blockIdx.x) < a.token_blocks;
  const int first = static_cast<int>(blockIdx.x) * a.tokens, n = mover ? min(a.tokens, r.S - first) : 0;
  const RowCopy copy(a.row_bytes);
  // (the rows wait where sixteen waves select: a thread has half the registers then)
  RowWork work(a, copy, mover ? first : 0, FORM == kHoldWide ? 0 : n);
  const bool marked = not_set_up(a);
  int e[K];
  float p[K];
  bool mem[K];
  uint32_t rank[K];
  {
    const Routed t = route_tile_token<K, GD, FORM>(r.gate, r.noise, tid, r.S, r.E, r.is_logits != 0, s_cnt);
    if (threadIdx.x >= kTile) return;
    e[0] = t.e0, p[0] = t.p0;
    if (K == 2) e[K - 1] = t.e1, p[K - 1] = t.p1;
  }
#pragma unroll
  for (int j = 0; j < K; ++j) {
    if (tid >= r.S) e[j] = -1;
    mem[j] = e[j] >= 0;
  }
  TileStart me;
  me.tile = 0u, me.epoch = 0u, me.spin = 0u, me.ok = true;
  tile_scan<K, false>(e, mem, r.E, me, r.ws, s_cnt, rank);
  const uint32_t* totals = s_cnt + kWavesPerTile * K * r.E;
  if (!mover) {
    // (turns are no more than rows of the buffer, which 31 bits count)
    const uint32_t chunks = static_cast<uint32_t>(a.tail_chunks), turns = chunks * static_cast<uint32_t>(r.E);
    for (uint32_t turn = blockIdx.x - static_cast<uint32_t>(a.token_blocks); turn < turns; turn += static_cast<uint32_t>(a.tail_blocks)) {
      const int x = static_cast<int>(turn / chunks);
      const int64_t total = static_cast<int64_t>(totals[x]) + (K == 2 ? totals[r.E + x] : 0u);
      clear_tail(a, x, tail_start(a, x, total, marked), static_cast<int>(turn - static_cast<uint32_t>(x) * chunks));
    }
    return;
  }
  if (tid < r.S) {
    int fe[K], fl[K];
    float g[K];
    if (K == 1) {
      const int used = (r.used_in && e[0] >= 0) ? r.used_in[e[0]] : 0;
      const int l = static_cast<int>(rank[0]);
      fl[0] = e[0] >= 0 ? l : 0;
      fe[0] = (e[0] < 0 || l >= r.C - used) ? -1 : e[0];
      g[0] = p[0];
    } else {
      const int e1 = e[0], e2 = e[K - 1];
      const int u1 = (r.used_in && e1 >= 0) ? r.used_in[e1] : 0, u2 = (r.used_in && e2 >= 0) ? r.used_in[e2] : 0;
      const Top2Place t = place_top2(e1, static_cast<int>(rank[0]), e2, static_cast<int>(rank[K - 1]), u1, u2, e2 >= 0 ? totals[e2] : 0u, r.E, r.C);
      fe[0] = t.e1, fl[0] = t.l1, fe[K - 1] = t.e2, fl[K - 1] = t.l2;
      // the raw values as a gate array holds them, normalised in fp32, rounded once
      const float g1 = t.e1 >= 0 ? round_gate(p[0], GD) : 0.f, g2 = t.e2 >= 0 ? round_gate(p[K - 1], GD) : 0.f;
      const float den = fmaxf(g1 + g2, 1.1920929e-07f);
      g[0] = g1 / den, g[K - 1] = g2 / den;
    }
    if (marked) {
#pragma unroll
      for (int j = 0; j < K; ++j) fe[j] = fl[j] = -1, g[j] = 0.f;
    }
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (tid >= first && tid < first + n) s_dest[j * kTile + tid - first] = buffer_row(a, fe[j], fl[j]);
      if (blockIdx.x == 0) {
        r.idx_out[j * r.S + tid] = fe[j];
        r.loc_out[j * r.S + tid] = fl[j];
        st_gate(r.gates_s, static_cast<size_t>(j) * r.S + tid, g[j], GD);
      }
    }
  }
  if (blockIdx.x == 0) store_totals<K>(r, totals, marked);
  if (FORM == kHoldWide) work.load(a, copy, first, n);
  __syncthreads();
  work.store<K>(a, copy, first, n, s_dest);
}

// A few tiles, behind route_count_kernel: a workgroup adds up the counts of the tiles before its own (and of all), finishes
// its tokens' routing, which nobody else reads or writes, and moves their rows.
template <int K>
__global__ __launch_bounds__(kTile) void encode_place_rows_kernel(EncodeArgs a) {
  extern __shared__ uint32_t s_sum[];  // [2][K * E]: before this tile, all tiles
  __shared__ int s_dest[K * kTile];
  const RouteArgs& r = a.r;
  const int tid = threadIdx.x, NC = K * r.E;
  uint32_t* s_before = s_sum;
  uint32_t* s_total = s_sum + NC;
  const bool marked = not_set_up(a);
  if (static_cast<int>(blockIdx.x) >= a.token_blocks) {
    // the totals of one expert
    const int tb = static_cast<int>(blockIdx.x) - a.token_blocks, x = tb / a.tail_blocks;
    const int PP = count_pairs(NC);
    uint32_t t = 0;
    for (int i = tid; i < K * r.ntiles; i += kTile) {
      const int c = K == 2 && i >= r.ntiles ? r.E + x : x;
      const uint64_t w = r.ws.desc[static_cast<size_t>(K == 2 && i >= r.ntiles ? i - r.ntiles : i) * PP + (c >> 1)];
      t += c & 1 ? static_cast<uint32_t>(w >> 32) & kEpochMask : static_cast<uint32_t>(w);
    }
    if (tid == 0) s_sum[0] = 0u;
    __syncthreads();
    if (t) atomicAdd(&s_sum[0], t);
    __syncthreads();
    const int64_t from = tail_start(a, x, s_sum[0], marked);
    for (int chunk = tb - x * a.tail_blocks; chunk < a.tail_chunks; chunk += a.tail_blocks) clear_tail(a, x, from, chunk);
    return;
  }
  const int first = static_cast<int>(blockIdx.x) * a.tokens, n = min(a.tokens, r.S - first);
  const RowCopy copy(a.row_bytes);
  RowWork work(a, copy, first, n);
  // the token of thread tid < n
  int e[K], l[K];
  float g[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    e[j] = -1, l[j] = 0, g[j] = 0.f;
    if (tid < n) {
      e[j] = r.idx_out[j * r.S + first + tid];
      l[j] = r.loc_out[j * r.S + first + tid];
      if (K == 2) g[j] = ld_gate(r.gates_s, static_cast<size_t>(j) * r.S + first + tid, r.gate_dtype);
    }
    if (e[j] >= r.E) e[j] = -1;
  }
  sum_tile_counts(r.ws, static_cast<uint32_t>(first / kTile), r.ntiles, NC, 0, s_before, s_total);
  if (tid < n) {
    const int s = first + tid;
    int fe[K], fl[K];
    if (K == 1) {
      const int used = (r.used_in && e[0] >= 0) ? r.used_in[e[0]] : 0;
      fl[0] = e[0] >= 0 ? static_cast<int>(s_before[e[0]]) + l[0] : 0;
      fe[0] = (e[0] < 0 || fl[0] >= r.C - used) ? -1 : e[0];
    } else {
      const int e1 = e[0], e2 = e[K - 1];
      const int r1 = (e1 >= 0 ? static_cast<int>(s_before[e1]) : 0) + l[0], r2 = (e2 >= 0 ? static_cast<int>(s_before[r.E + e2]) : 0) + l[K - 1];
      const int u1 = (r.used_in && e1 >= 0) ? r.used_in[e1] : 0, u2 = (r.used_in && e2 >= 0) ? r.used_in[e2] : 0;
      const Top2Place t = place_top2(e1, r1, e2, r2, u1, u2, e2 >= 0 ? s_total[e2] : 0u, r.E, r.C);
      fe[0] = t.e1, fl[0] = t.l1, fe[K - 1] = t.e2, fl[K - 1] = t.l2;
      const float g1 = t.e1 >= 0 ? g[0] : 0.f, g2 = t.e2 >= 0 ? g[K - 1] : 0.f;
      const float den = fmaxf(g1 + g2, 1.1920929e-07f);
      st_gate(r.gates_s, s, marked ? 0.f : g1 / den, r.gate_dtype);
      st_gate(r.gates_s, static_cast<size_t>(r.S) + s, marked ? 0.f : g2 / den, r.gate_dtype);
    }
    if (K == 1 && marked) st_gate(r.gates_s, s, 0.f, r.gate_dtype);
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (marked) fe[j] = fl[j] = -1;
      r.idx_out[j * r.S + s] = fe[j];
      r.loc_out[j * r.S + s] = fl[j];
      s_dest[j * kTile + tid] = buffer_row(a, fe[j], fl[j]);
    }
  }
  if (blockIdx.x == 0) store_totals<K>(r, s_total, marked);
  __syncthreads();
  work.store<K>(a, copy, first, n, s_dest);
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
// Which encodes are short.  (Separate kernels / this file's, us, bf16 rows, fp32 logits.)
//   One tile: every workgroup routes it, so the gate must be small or its rows short enough for a walk that the launches it
//   saves outweigh.  64 x 1024 top-2, 8 experts 9.1 / 4.6, 32 experts 9.7 / 5.9, 128 experts 15.6 / 11.6; 256 tokens, 128 experts
//   16.8 / 12.9; but 128 tokens, 256 experts 22.6 / 24.8 and 256 tokens, 512 experts 43 / 90.
//   A few tiles: a workgroup adds up the counts of all tiles, so there must be few; and what the saved launch gives is lost again
//   where long rows go to two places, which many short workgroups do better.  Buffers that no cache holds, 8 experts: top-1
//   2000 x 1024 9.4 / 7.5, 8192 x 1024 14.6 / 11.7, 8192 x 2048 22.4 / 19.9; top-2 4096 x 512 10.6 / 10.0, 4096 x 2048 17.5 / 19.4, 8192 x
//   4096 48.4 / 52.0.  64 tiles, top-1: x 256 10.1 / 9.5, x 512 13.3 / 13.6, x 2048 34.0 / 33.7; 128 tiles x 256 14.0 / 14.5.
//   Long top-1 rows: 40 MB of 8192 bytes 23.6 / 24.6, 50 MB 26.6 / 27.9, 62 MB 30.6 / 34; with 64 experts, whose separate routing takes
//   longer, 28.2 / 26.5, 34.7 / 34.2 and 35.2 / 36.0.
constexpr int64_t kTileGate = 16384, kTileExperts = 128;
constexpr int64_t kShortTiles = 32, kShortCounts = 4096;
constexpr size_t kShortRows2 = 12u << 20;  // bytes of token rows, top-2
static size_t short_rows1(int64_t E) { return static_cast<size_t>(E >= 32 ? 52 : 36) << 20; }  // ... top-1
// Workgroups that move rows: each takes twice the tokens while there are more than this.  Best are 1000 to 1700, and half of what just
// exceeds the limit is the worst case.  Arrays that no cache holds, tokens x bytes, us by workgroups (separate kernels): top-2 6510 x
// 1536 407 17.4, 814 14.9, 1628 14.5 (15.0); 3255 x 3072 407 18.1, 814 15.6, 1628 13.7 (15.1); 7812 x 1536 488 18.5, 977 15.8, 1953 17.4 (16.0);
// 2000 x 6000 500 18.8, 1000 16.9, 2000 17.5 (16.6); 1220 x 8192 610 15.0, 1220 13.0 (14.9); 5859 x 2048 732 15.4, 1465 15.5 (15.7); top-1 6666 x
// 6000 834 28.5, 1667 25.0 (24.4); 3333 x 6000 834 17.2, 1667 14.5, 3333 15.6 (17.1); 6510 x 3072 814 16.2, 1628 14.8, 3255 16.1 (16.6); 3662 x 8192
// 916 20.4, 1831 19.4, 3662 20.0 (19.4); 4882 x 4096 1221 14.0, 2441 15.3 (15.8).
constexpr int kShortBlocks1 = 2000, kShortBlocks2 = 1700;
// Tails.  A turn clears 32 KB, 16 rows at least.  Of one tile, every workgroup that clears has to route the tile first, so there
// are only as many as the movers leave CUs idle, each with several turns; a second one on a CU costs the routing again (256 x
// 1024 top-2, 128 experts, capacity 20: 10.9 us with 192 of them beside 64 movers, 15.9 with 256), and one per 16 rows, as many as
// the buffer has, made the capacity the bound: separate kernels / one workgroup per turn of 16 rows / now, us: 256 x 64 top-1, 128
// experts, capacity 256 14.2 / 39.4 / 7.8, 4096 33.6 / 530 / 18.2; 256 x 1024 top-2, 128 experts, capacity 256 28.7 / 58.9 / 20.2, 4096
// 209 / 744 / 204; 64 x 64 top-2, 128 experts, capacity 128 15.2 / 18.4 / 7.5; 1 x 1024 top-2, 512 experts 36.1 / 47.2 / 34.6.  (fp32 logits of
// more than 256 experts for 17 to 32 tokens run faster with two on a CU, 32 x 1024 top-1 23.2 / 26.9, and for 16 tokens slower,
// 35.0 / 26.6: not understood.)  Of a few tiles, a workgroup adds up its expert's counts: 8192 x 64 top-1, 64 experts, capacity 8192
// 31.7 / 52.5 / 19.4, 8192 x 1024, capacity 160 16.8 / 14.0 / 13.8.
constexpr int kShortTailRows = 16;
constexpr uint32_t kShortTailBytes = 32768;
constexpr int kCus = 256, kTileTails = 128;  // (movers on every CU: half as many again)
constexpr int kShortTails = 4096;            // of a few tiles, all experts together
constexpr int kShortPerLane = 2;  // granules per lane (one: 6000 x 1024 top-1 12.3 us against 10.9, top-2 16.8 against 13.7)

bool encode_is_short(const int32_t* used_in, const int32_t* used_out, int64_t S, int64_t E, int K, size_t row_bytes, bool force_lookback) {
  // (a caller that has used capacity updated in place gets the separate kernels: here every workgroup reads what the first writes)
  if (force_lookback || S < 1 || row_bytes == 0 || (used_in != nullptr && used_in == used_out)) return false;
  if (S <= kTile) return S * E <= kTileGate || E <= kTileExperts;
  const int64_t tiles = scan_num_tiles(S);
  return tiles <= kShortTiles && tiles * K * E <= kShortCounts && static_cast<size_t>(S) * row_bytes <= (K == 1 ? short_rows1(E) : kShortRows2);
}

hipError_t run_encode_short(const void* data, const void* gate, const void* noise, const int32_t* used_in, int S, int E, int C, int M,
                            int K, bool is_logits, int elem_bytes, int gate_dtype, bool tail, bool rows_at_used, void* gates_s,
                            int32_t* idx_out, int32_t* loc_out, int32_t* used_out, uint64_t* elems_out, void* out, void* ws,
                            hipStream_t st) {
  EncodeArgs a;
  RouteArgs& r = a.r;
  r.gate = gate, r.noise = K == 2 ? noise : nullptr, r.idx_in = nullptr, r.used_in = used_in, r.gates_s = gates_s;
  r.idx_out = idx_out, r.loc_out = loc_out, r.used_out = used_out, r.elems_out = elems_out, r.ws = scan_ws_view(ws);
  r.S = S, r.E = E, r.C = C, r.M = M, r.ntiles = static_cast<int>(scan_num_tiles(S)), r.is_logits = is_logits, r.gate_dtype = gate_dtype, r.seg_rows = 0;
  a.data = static_cast<const char*>(data), a.out = static_cast<char*>(out);
  a.row_bytes = static_cast<uint32_t>(M) * static_cast<uint32_t>(elem_bytes);
  const long units = a.row_bytes >= 16 ? (a.row_bytes + 15L) / 16 : a.row_bytes / 2;
  a.q = 0;
  while (a.q < 8 && (static_cast<long>(kShortPerLane) << a.q) < units) ++a.q;
  a.tokens = kTile >> a.q;
  while (a.tokens < kTile && (S + a.tokens - 1) / a.tokens > (K == 1 ? kShortBlocks1 : kShortBlocks2)) a.tokens *= 2;
  a.token_blocks = (S + a.tokens - 1) / a.tokens;
  a.tail_rows = std::max(kShortTailRows, static_cast<int>(kShortTailBytes / a.row_bytes));
  a.tail_chunks = tail ? (C + a.tail_rows - 1) / a.tail_rows : 0;
  const int64_t turns = static_cast<int64_t>(a.tail_chunks) * E;
  a.tail_blocks = static_cast<int>(r.ntiles == 1 ? std::min<int64_t>(turns, std::max(kCus - a.token_blocks, kTileTails)) : std::min(a.tail_chunks, std::max(kShortTails / E, 1)));
  a.rows_at_used = rows_at_used && used_in != nullptr;
  a.needs_setup = scan_form(r.ntiles, static_cast<int64_t>(K) * E, K) == kScanLookback;
  const unsigned blocks = static_cast<unsigned>(a.token_blocks + (r.ntiles == 1 ? a.tail_blocks : a.tail_blocks * E));
  const int NC = K * E;
  if (r.ntiles == 1) {
    const SelectLaunch sel = select_launch(gate_dtype, gate, r.noise, S, E, is_logits);
    const size_t lds = std::max(scan_lds_bytes(NC), sel.lds);
    LANCET_SELECT_SWITCH(gate_dtype, sel.form,
      if (K == 1) encode_tile_kernel<1, GD, FORM><<<blocks, sel.threads, lds, st>>>(a);
      else encode_tile_kernel<2, GD, FORM><<<blocks, sel.threads, lds, st>>>(a))
    return hipGetLastError();
  }
  const hipError_t err = run_route_count(r, K, st);
  if (err != hipSuccess) return err;
  const size_t lds = 2 * static_cast<size_t>(NC) * sizeof(uint32_t);
  if (K == 1) encode_place_rows_kernel<1><<<blocks, kTile, lds, st>>>(a);
  else encode_place_rows_kernel<2><<<blocks, kTile, lds, st>>>(a);
  return hipGetLastError();
}

}  // namespace lancet
