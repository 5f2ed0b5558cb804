// Batch-prioritised routing (raf.op.moe_encode_batch_prioritized): radix select instead of an argsort, then
// a position scan with two counter sets.
#include "launchers.hpp"
#include "select.hpp"
#include <algorithm>

namespace lancet {

// ---------------------------------------------------------------------------------------
// Batch-prioritised routing.
//   bpr_select_kernel : one workgroup per expert.  Finds, with a radix select of 10-bit digits on the
//                       order-preserving integer image of the fp32 priority, the C-th largest
//                       priority among the expert's tokens (threshold), how many ties at the
//                       threshold may stay (quota, lowest token ids first) and how many ties
//                       lie before the partition (ties_before).
//   bpr_scan_kernel   : tile scan over the partition with two counter sets (tokens above the
//                       threshold / tokens at the threshold); a token stays iff it is above,
//                       or at the threshold with global tie rank < quota; its location is
//                       above_before + min(tie_rank, quota) - min(ties_before, quota).
// Equivalent to the reference's stable descending argsort + keep-first-C + compaction
// (src/op/dialect/cuda/moe.cc:638-683, tutel_moe_dispatch.cu:259-363) without sorting.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t order_key(float x) {
  if (x == 0.f) x = 0.f;  // -0 and +0 compare equal in a float sort
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Everything the batch-prioritised routing keeps in the scan's workspace behind the descriptor table is a
// 64-bit word tagged "not a descriptor" (foreign_word), the value in the low half: tok[s] also carries the
// token's expert + 1 in the tag's low bits; par[0..2][e] = threshold, tie quota, ties before the partition,
// par[3][e] = tokens of the expert before the partition inside the tile of 256 tokens that holds its start.
// For the select kernel the prepare kernel also leaves every tile's keys grouped by expert, in token order
// (keys[tile][256], the token's place in its tile in the tag) and where each expert's group lies (groups[e][tile] = start | count << 16): an expert's
// workgroup then reads its own keys and one word per tile instead of the whole batch.
struct BprArgs {
  uint64_t* tok;         // [S0] expert and priority (gate value of the chosen expert) per token
  uint64_t* par;         // [4][E]
  uint64_t* keys;        // [ntiles0][256] order keys, grouped by expert inside a tile
  uint64_t* groups;      // [E][ntiles0]
  int ntiles0;           // tiles of the whole batch
  int S0, S, E, C, M;
  int part_lo;           // first token of the partition
  int ntiles;
  int seg_rows;          // place kernel: tiles per segment of the segment sums, 0 = there are none
  int placed_by_expert;  // the select kernel also places the tokens: no scan follows
  int gate_dtype;        // storage type of gates_s (and of the gate the priorities came from)
  void* gates_s;         // [S]
  int32_t* idx_out;      // [S]
  int32_t* loc_out;      // [S]
  int32_t* used_out;     // [E]
  uint64_t* elems_out;   // [E]
  ScanWs ws;
};

constexpr int kSelectThreads = 1024;

__device__ __forceinline__ int tok_expert(uint64_t w) { return static_cast<int>((w >> 32) & 0xffffu) - 1; }
__device__ __forceinline__ float tok_prio(uint64_t w) { return __uint_as_float(static_cast<uint32_t>(w)); }
__device__ __forceinline__ uint32_t par_value(const uint64_t* p) { return static_cast<uint32_t>(*p); }

// first choice and its gate value (or softmax probability) of every token of the batch
// (the priority is the gate value as gates_s will hold it: rounded to the gate type); the tile's keys grouped
// by expert
template <int GD, int FORM>
__global__ __launch_bounds__(kSelectThreadsOf<FORM>) void bpr_prepare_kernel(const void* gate, int is_logits, BprArgs a) {
  extern __shared__ uint32_t s_cnt[];
  const int tid = threadIdx.x;
  const uint32_t tile = blockIdx.x;
  const int s = static_cast<int>(tile) * kTile + tid;
  int cls[1] = {-1};
  uint32_t key = 0;
  const Routed r = route_tile_token<1, GD, FORM>(gate, nullptr, s, a.S0, a.E, is_logits != 0, s_cnt);
  if (threadIdx.x >= kTile) return;
  if (s < a.S0) {
    const float prio = round_gate(r.p0, GD);
    a.tok[s] = foreign_word(static_cast<uint32_t>(r.e0 + 1), __float_as_uint(prio));
    cls[0] = r.e0;
    key = order_key(prio);
  }
  const bool mem[1] = {cls[0] >= 0};
  uint32_t rank[1];
  TileStart me;
  me.tile = tile, me.epoch = 0u, me.spin = 0u, me.ok = true;
  tile_scan<1, false>(cls, mem, a.E, me, a.ws, s_cnt, rank);  // rank among the tile's tokens of the same expert
  __syncthreads();  // every wave has its ranks: rows of s_cnt can be reused
  // rows of s_cnt the scan without look-back leaves unused (zero): where each expert's group starts, and how many
  // of its tokens come before the partition
  const uint32_t* s_agg = s_cnt + kWavesPerTile * a.E;
  uint32_t* s_start = s_cnt + (kWavesPerTile + 1) * a.E;
  uint32_t* s_early = s_start + a.E;
  const bool holds_start = static_cast<int>(tile) == a.part_lo / kTile;
  if (tid < kWave) {
    // exclusive scan of the tile's counts over the experts: lane l owns `per` consecutive experts
    const int per = (a.E + kWave - 1) / kWave;
    uint32_t mine = 0;
    for (int i = 0; i < per; ++i) mine += (tid * per + i < a.E) ? s_agg[tid * per + i] : 0u;
    uint32_t inc = mine;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const uint32_t v = __shfl_up(inc, off, kWave);
      if (tid >= off) inc += v;
    }
    uint32_t run = inc - mine;
    for (int i = 0; i < per; ++i) {
      const int c = tid * per + i;
      if (c < a.E) {
        s_start[c] = run;
        run += s_agg[c];
      }
    }
  }
  if (holds_start && cls[0] >= 0 && s < a.part_lo) atomicAdd(&s_early[cls[0]], 1u);
  __syncthreads();
  if (cls[0] >= 0) a.keys[static_cast<size_t>(tile) * kTile + s_start[cls[0]] + rank[0]] = foreign_word(static_cast<uint32_t>(tid), key);
  if (a.placed_by_expert && s >= a.part_lo && s < a.part_lo + a.S) st_gate(a.gates_s, s - a.part_lo, cls[0] >= 0 ? round_gate(r.p0, GD) : 0.f, GD);
  for (int c = tid; c < a.E; c += kTile) {
    a.groups[static_cast<size_t>(c) * a.ntiles0 + tile] = foreign_word(0u, s_start[c] | (s_agg[c] << 16));
    if (holds_start) a.par[3 * a.E + c] = foreign_word(0u, s_early[c]);
  }
}

// Keys of one expert kept in LDS (128 KB): the largest power of two that leaves room for the tiles' positions.  An
// expert that half of a batch of 65536 tokens chose still fits.
constexpr int kSelectKeys = 32768;
constexpr int kSelectTiles = 4096;  // tiles whose group positions fit in LDS (16 KB): batches up to 1M tokens
// Tokens of a batch up to which an expert's workgroup also places its tokens, which saves the two launches of the scan; in longer
// batches the expert that most tokens chose is placed by one CU, store by store.  moe_encode_batch_prioritized of rows of 32
// bytes, scan / placed, us: 64 tokens on 8 experts 14.9 / 12.6, 512 on 16 17.3 / 15.0, 1024 on 64 19.8 / 15.1, 2048 on 4, nearly all on
// one, 18.0 / 17.7; 4096 on 64 22.9 / 18.6, but nearly all on one of two 18.5 / 20.6, and 32768 on 64, some hot, 35.0 / 42.6.
constexpr int kPlaceTokens = 2048;
static_assert(kPlaceTokens <= kSelectKeys, "the keys lie in LDS");
constexpr int kSelectBits = 10;     // digit of the radix select: one histogram bin per thread
static_assert((1 << kSelectBits) == kSelectThreads, "a thread owns one bin");

// exclusive scan over the kSelectThreads values of a workgroup; *total = their sum.  s_wave: 16 words of LDS.
__device__ __forceinline__ uint32_t select_block_scan(uint32_t v, uint32_t* s_wave, uint32_t* total) {
  const int lane = lane_id(), w = threadIdx.x / kWave;
  uint32_t inc = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t u = __shfl_up(inc, off, kWave);
    if (lane >= off) inc += u;
  }
  __syncthreads();  // s_wave may still be read from an earlier call
  if (lane == kWave - 1) s_wave[w] = inc;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < kSelectThreads / kWave; ++k) {
    const uint32_t t = s_wave[k];
    before += (k < w) ? t : 0u;
    all += t;
  }
  *total = all;
  return before + inc - v;
}

// f(key's word, tile, position) for every key of the expert, position = its place in token order, from the prepare kernel's groups.
// A group is read by 2^q neighbouring lanes, q by the expert's mean keys per tile, four loads of a lane in flight:
// s_pos holds the position of a tile's first key in the low 22 bits and the start of its group inside the tile above
// them, so nothing is searched for.  (A lane that found the tile of its key by bisection over the positions spent most of
// the kernel on it: 12 dependent LDS reads per key.)
template <typename F>
__device__ __forceinline__ void walk_groups(const BprArgs& a, const uint32_t* s_pos, uint32_t count, int q, F f) {
  const uint32_t width = 1u << q;
  const uint32_t sub = threadIdx.x & (width - 1u);
  for (int t = static_cast<int>(threadIdx.x >> q); t < a.ntiles0; t += kSelectThreads >> q) {
    const uint32_t w = s_pos[t];
    const uint32_t pos = w & 0x3fffffu;
    const uint32_t n = (t + 1 < a.ntiles0 ? s_pos[t + 1] & 0x3fffffu : count) - pos;
    const uint64_t* group = a.keys + static_cast<size_t>(t) * kTile + (w >> 22);
    for (uint32_t i = sub; i < n; i += 4u * width) {
      uint64_t k[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) k[j] = i + j * width < n ? group[i + j * width] : 0ull;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (i + j * width < n) f(k[j], t, pos + i + j * width);
    }
  }
}

// One workgroup per expert.  What bounds it is, in long batches, the one expert that most tokens chose, whose keys a single
// CU reads and counts; in short ones the barriers of its 1024 threads, of which a digit takes six.  The digits start below
// the leading bits that all keys share (probabilities have two or three exponents, so a digit that starts at bit 31 puts
// every key into the same few bins, whose LDS atomics then run one after the other).  As soon as no more keys than a wave has
// lanes share what is found of the threshold, which is mostly after one digit, they are compared with one another.  32768
// tokens on 64 experts of which a few are hot (top-1, most keys on one expert): four 8-bit digits from bit 31 on 78 us, three
// of 10 bits 18.5.  moe_encode_batch_prioritized as a whole, the same two and with the keys compared after the first digit:
// 256 tokens on 16 experts 17.1 / 18.2 / 15.6 us, 1024 on 64 20.5 / 21.4 / 18.7.
//
// PLACE (short batches, whose keys all fit in LDS): the workgroup goes on to place its expert's tokens: two scans over the keys
// in token order, ties and kept ones, give every kept token its location, and a second walk over the groups, which name the
// tokens, writes them.
template <bool PLACE>
__global__ __launch_bounds__(kSelectThreads) void bpr_select_kernel(BprArgs a) {
  __shared__ uint32_t s_keys[kSelectKeys];
  __shared__ uint32_t s_pos[kSelectTiles];
  __shared__ uint32_t hist[1 << kSelectBits];
  __shared__ uint32_t s_wave[kSelectThreads / kWave];
  __shared__ uint32_t s_prefix, s_need, s_count, s_min, s_max, s_bin, s_few;
  __shared__ uint32_t s_thr, s_quota, s_front, s_kept;  // PLACE: what was selected
  const int e = blockIdx.x;
  const int tid = threadIdx.x;
  // The expert's keys, in token order.  Up to kSelectTiles tiles, the prepare kernel's groups say where they are:
  // positions by a scan over the tiles, then the keys themselves into LDS (or, more than LDS holds, fetched again
  // in every pass).  Longer batches are read whole, once per pass.
  const bool grouped = a.ntiles0 <= kSelectTiles;
  uint32_t count = 0, nfront = 0;
  if (tid == 0) {
    s_count = 0;
    s_few = 0;
    s_min = 0xffffffffu;
    s_max = 0u;
    s_kept = 0;
    s_front = 0;
  }
  if (grouped) {
    uint32_t carry = 0;
    const int tstart = a.part_lo / kTile;  // the tile that holds the partition's first token
    const uint32_t early = a.S0 > 0 ? par_value(a.par + 3 * a.E + e) : 0u;
    for (int base = 0; base < a.ntiles0; base += kSelectThreads) {
      const int t = base + tid;
      const uint32_t g = t < a.ntiles0 ? static_cast<uint32_t>(a.groups[static_cast<size_t>(e) * a.ntiles0 + t]) : 0u;
      uint32_t total;
      const uint32_t pos = carry + select_block_scan(g >> 16, s_wave, &total);
      if (t < a.ntiles0) s_pos[t] = pos | ((g & 0xffffu) << 22);
      carry += total;
    }
    __syncthreads();
    count = carry;
    nfront = a.S0 > 0 ? (s_pos[tstart] & 0x3fffffu) + early : 0u;
  } else {
    __syncthreads();
    uint32_t local = 0;
    for (int s = tid; s < a.S0; s += kSelectThreads) local += (tok_expert(a.tok[s]) == e);
    if (local) atomicAdd(&s_count, local);
    __syncthreads();
    count = s_count;
  }
  const bool none = a.C <= 0, all = !none && count <= static_cast<uint32_t>(a.C);
  if (!PLACE && (none || all)) {
    // nothing fits: no key is above the largest threshold and the tie quota is zero; everything fits: every key is above
    // threshold 0 or ties with it under an unlimited quota
    if (tid == 0) {
      a.par[e] = foreign_word(0u, none ? 0xffffffffu : 0u);
      a.par[a.E + e] = foreign_word(0u, none ? 0u : 0x7fffffffu);
      a.par[2 * a.E + e] = foreign_word(0u, 0u);
    }
    return;
  }
  const bool in_lds = grouped && count <= kSelectKeys;
  int q = 0;
  while (q < 6 && static_cast<uint64_t>(a.ntiles0) << q < count) ++q;
  // f(key, whether its token lies before the partition) for all keys
  const auto every_key = [&](auto f) {
    if (in_lds) {
      for (uint32_t i = tid; i < count; i += kSelectThreads) f(s_keys[i], i < nfront);
    } else if (grouped) {
      walk_groups(a, s_pos, count, q, [&](uint64_t w, int, uint32_t pos) { f(static_cast<uint32_t>(w), pos < nfront); });
    } else {
      for (int s = tid; s < a.S0; s += kSelectThreads) {
        const uint64_t t = a.tok[s];
        if (tok_expert(t) == e) f(order_key(tok_prio(t)), s < a.part_lo);
      }
    }
  };
  const auto select = [&] {
    uint32_t lo = 0xffffffffu, hi = 0u;
    if (in_lds) {
      walk_groups(a, s_pos, count, q, [&](uint64_t w, int, uint32_t pos) {
        const uint32_t k = static_cast<uint32_t>(w);
        s_keys[pos] = k;
        lo = min(lo, k), hi = max(hi, k);
      });
    } else {
      every_key([&](uint32_t k, bool) { lo = min(lo, k), hi = max(hi, k); });
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      lo = min(lo, static_cast<uint32_t>(__shfl_xor(lo, off, kWave)));
      hi = max(hi, static_cast<uint32_t>(__shfl_xor(hi, off, kWave)));
    }
    if (lane_id() == 0) {
      atomicMin(&s_min, lo);
      atomicMax(&s_max, hi);
    }
    if (tid == 0) s_need = static_cast<uint32_t>(a.C);
    __syncthreads();
    // digits from the highest bit in which two keys differ; `left` bits are still to be found
    int left = s_min == s_max ? 0 : 32 - __clz(s_min ^ s_max);
    uint32_t prefix = left == 32 ? 0u : s_min >> left;
    uint32_t open = count;  // keys that share what is found of the threshold
    while (left > 0 && open > kWave) {
      const int bits = min(left, kSelectBits);
      const int shift = left - bits;
      const uint32_t digits = (1u << bits) - 1u;
      hist[tid] = 0;
      __syncthreads();
      const uint32_t need = s_need;
      every_key([&](uint32_t k, bool) {
        if (left == 32 || (k >> left) == prefix) atomicAdd(&hist[(k >> shift) & digits], 1u);
      });
      __syncthreads();
      // the digit that holds the need-th largest of the keys counted, and what is needed inside it: bins in descending
      // order, one per thread
      const uint32_t bin = static_cast<uint32_t>(kSelectThreads - 1 - tid);
      const uint32_t h = hist[bin];
      uint32_t total;
      const uint32_t above = select_block_scan(h, s_wave, &total);
      // (fewer keys than needed does not happen with consistent counts: digit 0 takes what is left)
      if ((above < need && need <= above + h) || (bin == 0u && total < need)) {
        s_need = need - above;
        s_prefix = (left == 32 ? 0u : prefix << bits) | bin;
        s_bin = h;
      }
      __syncthreads();
      prefix = s_prefix;
      open = s_bin;
      left = shift;
    }
    if (left > 0) {
      // no more keys than a wave has lanes: it compares them with one another, and counts the threshold's equals that
      // precede the partition on the way
      every_key([&](uint32_t k, bool early) {
        if (left == 32 || (k >> left) == prefix) {
          const uint32_t at = atomicAdd(&s_few, 1u);
          hist[at] = k;
          hist[kWave + at] = early;
        }
      });
      __syncthreads();
      if (tid < static_cast<int>(open)) {
        const uint32_t mine = hist[tid];
        uint32_t above = 0, same = 0, front = 0;
        for (uint32_t i = 0; i < open; ++i) {
          above += hist[i] > mine;
          same += hist[i] == mine;
          front += (hist[i] == mine) & hist[kWave + i];
        }
        const uint32_t need = s_need;
        if (above < need && need <= above + same) {  // equal keys write the same words
          if (PLACE) {
            s_thr = mine;
            s_quota = need - above;
          } else {
            a.par[e] = foreign_word(0u, mine);
            a.par[a.E + e] = foreign_word(0u, need - above);
            a.par[2 * a.E + e] = foreign_word(0u, front);
          }
        }
      }
      return;
    }
    if (PLACE) {
      if (tid == 0) {
        s_thr = prefix;
        s_quota = s_need;
      }
      return;
    }
    const uint32_t thr = prefix;
    // ties that precede the partition
    if (a.part_lo > 0) {
      uint32_t local = 0;
      every_key([&](uint32_t k, bool early) { local += early && k == thr; });
      if (!grouped && tid == 0) s_count = 0;  // held the expert's count
      __syncthreads();
      if (local) atomicAdd(&s_count, local);
      __syncthreads();
    }
    if (tid == 0) {
      a.par[e] = foreign_word(0u, thr);
      a.par[a.E + e] = foreign_word(0u, s_need);
      a.par[2 * a.E + e] = foreign_word(0u, a.part_lo > 0 ? s_count : 0u);
    }
  };
  if (!none && !all) select();
  if (!PLACE) return;

  // ---- the tokens' places -----------------------------------------------------------------------------------------
  __syncthreads();
  if (!none && !all) {
    // a thread owns consecutive keys, an odd number of them (LDS banks): how many tie with the threshold before them, which of
    // them stay, how many stay before
    const uint32_t thr = s_thr, quota = s_quota;
    const uint32_t per = (count + kSelectThreads - 1) / kSelectThreads | 1u, lo = min(count, tid * per), hi = min(count, lo + per);
    uint32_t ties = 0, total;
    for (uint32_t p = lo; p < hi; ++p) ties += s_keys[p] == thr;
    ties = select_block_scan(ties, s_wave, &total);
    const uint32_t first_tie = ties;
    uint32_t kept = 0;
    for (uint32_t p = lo; p < hi; ++p) {
      const uint32_t k = s_keys[p];
      kept += k > thr || (k == thr && ties < quota);
      ties += k == thr;
    }
    uint32_t before = select_block_scan(kept, s_wave, &total);
    ties = first_tie;
    for (uint32_t p = lo; p < hi; ++p) {
      const uint32_t k = s_keys[p];
      const bool stays = k > thr || (k == thr && ties < quota);
      ties += k == thr;
      if (p == nfront) s_front = before;
      s_keys[p] = stays ? before : 0xffffffffu;
      before += stays;
    }
    if (tid == 0 && nfront >= count) s_front = total;
    __syncthreads();
  }
  const uint32_t front = all ? nfront : s_front;
  uint32_t kept = 0;
  walk_groups(a, s_pos, count, q, [&](uint64_t w, int t, uint32_t pos) {
    const int sl = t * kTile + static_cast<int>((w >> 32) & 0xffu) - a.part_lo;
    if (sl < 0 || sl >= a.S) return;
    const uint32_t place = none ? 0xffffffffu : all ? pos : s_keys[pos];
    const bool stays = place != 0xffffffffu;
    a.idx_out[sl] = stays ? e : -1;
    a.loc_out[sl] = stays ? static_cast<int>(place - front) : -1;
    kept += stays;
  });
  if (kept) atomicAdd(&s_kept, kept);
  __syncthreads();
  if (tid == 0) {
    a.used_out[e] = static_cast<int32_t>(s_kept);
    a.elems_out[e] = static_cast<uint64_t>(s_kept) * static_cast<uint64_t>(a.M);
  }
}

__global__ __launch_bounds__(kTile) void bpr_scan_kernel(BprArgs a) {
  extern __shared__ uint32_t s_cnt[];
  const int tid = threadIdx.x;
  const TileStart me = tile_begin(a.ws, a.ntiles);
  const uint32_t tile = me.tile;
  const int sl = static_cast<int>(tile) * kTile + tid;  // token inside the partition
  const bool valid = sl < a.S;
  if (!me.ok) {
    if (valid) {
      a.idx_out[sl] = -1;
      a.loc_out[sl] = -1;
      st_gate(a.gates_s, sl, 0.f, a.gate_dtype);
    }
    if (blockIdx.x == 0) {
      for (int c = tid; c < a.E; c += kTile) {
        a.used_out[c] = -1;
        a.elems_out[c] = 0;
      }
    }
    return;
  }
  int cls[2] = {-1, -1};
  bool mem[2] = {false, false};
  float prio = 0.f;
  if (valid) {
    const uint64_t t = a.tok[a.part_lo + sl];
    const int e = tok_expert(t);
    prio = tok_prio(t);
    if (e >= 0 && e < a.E) {
      const uint32_t k = order_key(prio);
      const uint32_t thr = par_value(a.par + e);
      cls[0] = cls[1] = e;
      mem[0] = k > thr;   // above the threshold: always stays
      mem[1] = k == thr;  // at the threshold: stays while the quota lasts
    }
  }
  uint32_t rank[2];
  const bool poisoned = tile_scan<2>(cls, mem, a.E, me, a.ws, s_cnt, rank);
  if (valid) {
    int idx = -1, loc = -1;
    if (cls[0] >= 0 && !poisoned) {
      const int e = cls[0];
      const int64_t q = static_cast<int32_t>(par_value(a.par + a.E + e));
      const int64_t tb = static_cast<int32_t>(par_value(a.par + 2 * a.E + e));
      const int64_t tie_rank = tb + rank[1];
      if (mem[0] || (mem[1] && tie_rank < q)) {
        idx = e;
        loc = static_cast<int>(static_cast<int64_t>(rank[0]) + min(tie_rank, q) - min(tb, q));
      }
    }
    a.idx_out[sl] = idx;
    a.loc_out[sl] = loc;
    st_gate(a.gates_s, sl, prio, a.gate_dtype);
  }
  if (static_cast<int>(tile) == a.ntiles - 1) {
    const uint32_t* s_agg = s_cnt + kWavesPerTile * 2 * a.E;
    const uint32_t* s_base = s_agg + 2 * a.E;
    for (int c = tid; c < a.E; c += kTile) {
      const int64_t q = static_cast<int32_t>(par_value(a.par + a.E + c));
      const int64_t tb = static_cast<int32_t>(par_value(a.par + 2 * a.E + c));
      const int64_t above = static_cast<int64_t>(s_base[c]) + s_agg[c];
      const int64_t ties = static_cast<int64_t>(s_base[a.E + c]) + s_agg[a.E + c];
      const int64_t kept = above + min(tb + ties, q) - min(tb, q);
      const int64_t uo = min(kept, static_cast<int64_t>(a.C));
      a.used_out[c] = poisoned ? -1 : static_cast<int32_t>(uo);
      a.elems_out[c] = poisoned ? 0 : static_cast<uint64_t>(uo * a.M);
    }
  }
  tile_end(a.ws, me, a.ntiles, 2 * a.E);
}

// ---- the same scan as two or three kernels that wait for nothing (scan_form) ---------------------------------
// class and membership of a partition token in the two counter sets, from its word and the expert's threshold
struct BprClass {
  int e;        // expert, -1 = none
  bool above;   // above the threshold: always stays
  bool tie;     // at the threshold: stays while the quota lasts
  float prio;
};
__device__ __forceinline__ BprClass bpr_classify(const BprArgs& a, int sl) {
  BprClass c = {-1, false, false, 0.f};
  const uint64_t t = a.tok[a.part_lo + sl];
  const int e = tok_expert(t);
  c.prio = tok_prio(t);
  if (e >= 0 && e < a.E) {
    const uint32_t k = order_key(c.prio);
    const uint32_t thr = par_value(a.par + e);
    c.e = e;
    c.above = k > thr;
    c.tie = k == thr;
  }
  return c;
}

// bpr_count_kernel: ranks inside the tile in both counter sets (left in loc_out, 16 bits each: a tile has 256
// tokens), the tile's counts -> table.
__global__ __launch_bounds__(kTile) void bpr_count_kernel(BprArgs a) {
  extern __shared__ uint32_t s_cnt[];
  const uint32_t tile = blockIdx.x;
  const int sl = static_cast<int>(tile) * kTile + threadIdx.x;
  const bool valid = sl < a.S;
  int cls[2] = {-1, -1};
  bool mem[2] = {false, false};
  if (valid) {
    const BprClass c = bpr_classify(a, sl);
    cls[0] = cls[1] = c.e;
    mem[0] = c.above;
    mem[1] = c.tie;
  }
  uint32_t rank[2];
  TileStart me;
  me.tile = tile, me.epoch = 0u, me.spin = 0u, me.ok = true;
  tile_scan<2, false>(cls, mem, a.E, me, a.ws, s_cnt, rank);
  store_tile_counts(a.ws, tile, 2 * a.E, s_cnt);
  if (valid) a.loc_out[sl] = static_cast<int>(rank[0] | (rank[1] << 16));
}

// bpr_place_kernel: adds what the tiles before counted and finishes the tile's tokens (what bpr_scan_kernel does
// after its look-back).
__global__ __launch_bounds__(kTile) void bpr_place_kernel(BprArgs a) {
  extern __shared__ uint32_t s_sum[];  // [2][2E]: before this tile, all tiles
  const int NC = 2 * a.E;
  uint32_t* s_before = s_sum;
  uint32_t* s_total = s_sum + NC;
  const uint32_t tile = blockIdx.x;
  sum_tile_counts(a.ws, tile, a.ntiles, NC, a.seg_rows, s_before, s_total);
  const int sl = static_cast<int>(tile) * kTile + threadIdx.x;
  if (sl < a.S) {
    const BprClass c = bpr_classify(a, sl);
    int idx = -1, loc = -1;
    if (c.e >= 0) {
      const uint32_t packed = static_cast<uint32_t>(a.loc_out[sl]);
      const int64_t q = static_cast<int32_t>(par_value(a.par + a.E + c.e));
      const int64_t tb = static_cast<int32_t>(par_value(a.par + 2 * a.E + c.e));
      const int64_t above_before = static_cast<int64_t>(s_before[c.e]) + (packed & 0xffffu);
      const int64_t tie_rank = tb + s_before[a.E + c.e] + (packed >> 16);
      if (c.above || (c.tie && tie_rank < q)) {
        idx = c.e;
        loc = static_cast<int>(above_before + min(tie_rank, q) - min(tb, q));
      }
    }
    a.idx_out[sl] = idx;
    a.loc_out[sl] = loc;
    st_gate(a.gates_s, sl, c.prio, a.gate_dtype);
  }
  if (tile == 0) {
    for (int c = threadIdx.x; c < a.E; c += kTile) {
      const int64_t q = static_cast<int32_t>(par_value(a.par + a.E + c));
      const int64_t tb = static_cast<int32_t>(par_value(a.par + 2 * a.E + c));
      const int64_t kept = static_cast<int64_t>(s_total[c]) + min(tb + static_cast<int64_t>(s_total[a.E + c]), q) - min(tb, q);
      const int64_t uo = min(kept, static_cast<int64_t>(a.C));
      a.used_out[c] = static_cast<int32_t>(uo);
      a.elems_out[c] = static_cast<uint64_t>(uo * a.M);
    }
  }
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
size_t bpr_workspace_bytes(int64_t S0, int64_t S, int64_t E) {
  // descriptor table of the partition's scan | tok[S0] | par[4][E] | keys[tiles of the batch][256] | groups[E][tiles]
  const size_t t0 = static_cast<size_t>(scan_num_tiles(S0));
  return scan_workspace_bytes(S, E, 2) +
         (static_cast<size_t>(S0) + 4 * static_cast<size_t>(E) + t0 * kTile + static_cast<size_t>(E) * t0) * 8;
}

hipError_t run_bpr_route(const void* gate, int S0, int E, int C, int M, int n_partitions,
                         int partition_id, bool is_logits, int gate_dtype, void* gates_s, int32_t* idx_out,
                         int32_t* loc_out, int32_t* used_out, uint64_t* elems_out, void* ws,
                         hipStream_t st, bool force_lookback) {
  const int S = S0 / n_partitions;
  BprArgs a;
  a.S0 = S0;
  a.S = S;
  a.E = E;
  a.C = C;
  a.M = M;
  a.part_lo = partition_id * S;
  a.ntiles = static_cast<int>(scan_num_tiles(S));
  a.ws = scan_ws_view(ws);
  a.tok = reinterpret_cast<uint64_t*>(static_cast<char*>(ws) + scan_workspace_bytes(S, E, 2));
  a.par = a.tok + S0;
  a.ntiles0 = static_cast<int>(scan_num_tiles(S0));
  a.keys = a.par + 4 * static_cast<size_t>(E);
  a.groups = a.keys + static_cast<size_t>(a.ntiles0) * kTile;
  a.gates_s = gates_s;
  a.gate_dtype = gate_dtype;
  a.idx_out = idx_out;
  a.loc_out = loc_out;
  a.used_out = used_out;
  a.elems_out = elems_out;
  hipError_t err = hipSuccess;
  a.placed_by_expert = !force_lookback && S0 <= kPlaceTokens;
  // (an empty batch still runs one tile, which leaves empty groups for the select kernel)
  const SelectLaunch sel = select_launch(gate_dtype, gate, nullptr, S0, E, is_logits);
  LANCET_SELECT_SWITCH(gate_dtype, sel.form, (bpr_prepare_kernel<GD, FORM><<<a.ntiles0, sel.threads, std::max(scan_lds_bytes(E), sel.lds), st>>>(gate, is_logits, a)))
  err = hipGetLastError();
  if (err != hipSuccess) return err;
  if (a.placed_by_expert) {
    bpr_select_kernel<true><<<E, kSelectThreads, 0, st>>>(a);
    return hipGetLastError();
  }
  bpr_select_kernel<false><<<E, kSelectThreads, 0, st>>>(a);
  err = hipGetLastError();
  if (err != hipSuccess) return err;
  a.seg_rows = 0;
  const ScanForm form = scan_form(a.ntiles, 2 * static_cast<int64_t>(E), 2, force_lookback);
  if (form != kScanLookback) {
    bpr_count_kernel<<<a.ntiles, kTile, scan_lds_bytes(2 * E), st>>>(a);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    if (form == kScanCountSegPlace) {
      a.seg_rows = seg_rows(a.ntiles);
      err = run_scan_segsum(ws, a.ntiles, 2 * E, a.seg_rows, st);
      if (err != hipSuccess) return err;
    }
    bpr_place_kernel<<<a.ntiles, kTile, 4 * static_cast<size_t>(E) * sizeof(uint32_t), st>>>(a);
    return hipGetLastError();
  }
  bpr_scan_kernel<<<a.ntiles, kTile, scan_lds_bytes(2 * E), st>>>(a);
  return hipGetLastError();
}

}  // namespace lancet
