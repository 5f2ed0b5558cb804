// Gate gradient of moe_encode as a whole: from the gradient of the op's OUTPUT gates_s back to the [S,E] array
// the op was given, through everything the op does to a gate value on the way:
//   top_k = 1, probabilities   nothing: grad[s, idx] = dy            (encode_backward_gate_kernel,
//                              src/op/dialect/cuda/kernels/tutel_moe_dispatch.cu:96-105; wired by
//                              src/op/grad/moe.cc:30-58)
//   top_k = 2                  the normalisation g_k / max(g_1 + g_2, eps) of the two kept values
//                              (docker/resources/sharded_moe.py:304-312; the clamp passes no gradient to the sum
//                              below eps)
//   LANCET_GATE_IS_LOGITS      the softmax the op fuses in front of the selection (sharded_moe.py:260):
//                              d x[e] = p[e] * (d p[e] - sum_j p[i_j] * d p[i_j])
// Probabilities of a 16-bit softmax are taken as computed (fp32), not as a 16-bit gates_s array would hold them:
// the difference is below that type's own rounding.  Dropped slots carry no gradient (their mask is zero,
// sharded_moe.py:296-297,306-307).  One launch: four lanes per token form the token's few scalars (row maximum,
// 1 / sum of exponentials, the two slot gradients), then the workgroup writes its 64 tokens' block of the
// result in memory order, every element once.
#include "launchers.hpp"
#include "select.hpp"
#include <algorithm>
#include <type_traits>

namespace lancet {

struct GateGradArgs {
  const void* dy;        // [K*S] gradient of gates_s
  const void* gate;      // [S,E] the forward's gate input (may be null for top-1 on probabilities)
  const int32_t* idx;    // [K*S] expert per slot after the drop (row 0 of indices_locations)
  void* out;             // [S,E]
  int S, E;
};

// How a workgroup writes its block of the result.
enum GateGradBlock {
  kValues = 0,      // value by value
  kGranules = 1,    // in granules, which rows are whole ones of
  kCutGranules = 2  // in granules that rows end inside of
};

// What bounds it is its length: two dependent round trips to memory, the exponentials of a row's lanes, and, in a kernel of 3 us,
// the code itself: one kernel for logits and probabilities, and for every way to write a block, fetched more of it than it ran.
// Rows that are not whole granules value by value / all rows in granules, one such kernel for both / now, us: 8192 x 60 bf16 top-2 logits 11.8 / 7.0 / 5.2, 8192 x 128 fp32 12.9 / 10.3 / 7.8,
// 65536 x 128 bf16 probabilities top-1 7.2 / 7.7 / 6.7, 65536 x 256 fp32 top-1 logits 37.8 / 33.9 / 32.8, 8192 x 4 bf16 top-2 3.5 / 4.6 / 3.2,
// 131072 x 10 bf16 top-2 8.4 / 12.3 / 8.0.  856 shapes of 500 to 131072 tokens and 2 to 512 experts: 0.82 of the first, 0.83 of the second.

// A token's row is walked by kSub lanes, each taking every kSub-th 16-byte granule (or element), two at a time, with the
// maximum and the sum of exponentials kept together and rescaled when a larger value comes; the lanes' pairs are then
// merged.  Few tokens per workgroup and few loads per lane: the launch is short (a 65536 x 32 gate is 8 MB) and
// only gets up to the memory system's speed when many waves are in flight.
constexpr int kSub = 4;                      // lanes per token
constexpr int kGradTokens = kTile / kSub;    // tokens per workgroup
// Rows of fewer granules than lanes are read value by value, so that all lanes have some, and as many at a time as the row has, each
// of which costs an exponential: 131072 x 10 bf16 top-1 6.9 us, in granules 9.8; 131072 x 2 top-2 5.5, always four values 6.3.
constexpr int kShortValues = 4;

// Maximum and sum of exponentials of a row WITHOUT the entries that carry a slot gradient: with those the sum would
// hide how far a selected probability is from 1 (1 - p = rest / sum loses every digit to rounding once the row is
// peaked; kept apart it is exact to a few ulp, and with it the gradient p (1 - p) dy of a saturated gate).  The values come a few
// granules at a time, those left out as -inf, whose term is zero.
struct MaxSum {
  float top = -INFINITY, sum = 0.f;
  template <int N, bool FIRST = false>  // FIRST: nothing has been added before
  __device__ __forceinline__ void add(const float (&f)[N]) {
    float m = top;
#pragma unroll
    for (int i = 0; i < N; ++i) m = fmaxf(m, f[i]);
    const float ref = m == -INFINITY ? 0.f : m;  // nothing but -inf so far: every term is zero
    float s = FIRST ? 0.f : sum * expf(top - ref);
#pragma unroll
    for (int i = 0; i < N; ++i) s += expf(f[i] - ref);
    sum = s;
    top = m;
  }
};

// per-token scalars of a workgroup's tokens, in LDS
struct GateGradTile {
  int i1[kGradTokens], i2[kGradTokens];      // experts that receive a slot gradient (-1: none)
  // factor of the entry of expert i1 / i2 / of every other expert: the gradient with respect to that array entry
  // (probabilities), or what p[e] is multiplied with (logits: d_j (1 - p_j) - p_other d_other, and -sum_j p_j d_j)
  float c1[kGradTokens], c2[kGradTokens], rest[kGradTokens];
  float top[kGradTokens], inv[kGradTokens];  // logits: row maximum and 1 / sum_e exp(x - max)
};

template <int K, int GD, bool LOGITS, int BLOCK>
__global__ __launch_bounds__(kTile) void encode_dgate_kernel(GateGradArgs a) {
  __shared__ GateGradTile sh;
  constexpr size_t gb = GD == LANCET_F32 ? 4 : 2;
  constexpr int V = 16 / gb;
  const int tid = threadIdx.x;
  const int first = blockIdx.x * kGradTokens;
  const int t = tid / kSub, sub = tid % kSub;
  const int s = min(first + t, a.S - 1);  // lanes past the batch repeat its last token (their result is not stored)
  // ---- kSub lanes per token ---------------------------------------------------------------------------------
  {
    const char* row = static_cast<const char*>(a.gate) + static_cast<size_t>(s) * a.E * gb;
    int e[2] = {-1, -1};
    float dy[2] = {0.f, 0.f}, raw[2] = {0.f, 0.f};
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int x = a.idx[static_cast<size_t>(j) * a.S + s];
      if (x >= 0 && x < a.E) {
        e[j] = x;
        dy[j] = ld_gate(a.dy, static_cast<size_t>(j) * a.S + s, GD);
        if (K == 2 || LOGITS) raw[j] = gate_at<GD>(row, x);  // top-1 on probabilities needs no gate
      }
    }
    float top = 0.f, inv = 1.f, rest = 0.f;  // rest: sum of exponentials of the entries without a slot gradient
    float g[2] = {raw[0], raw[1]};           // the two kept probabilities (0 for a dropped slot)
    if (LOGITS) {
      MaxSum ms;
      const int n = (a.E + V - 1) / V;  // granules of the row
      if (n < kSub && a.E <= kSub * kShortValues) {
        const auto values = [&](auto per_lane) {
          float f[per_lane.value];
#pragma unroll
          for (int i = 0; i < per_lane.value; ++i) {
            const int j = sub + i * kSub;
            const float x = gate_at<GD>(row, min(j, a.E - 1));
            f[i] = ((j < a.E) & (j != e[0]) & (j != e[1])) ? x : -INFINITY;
          }
          ms.template add<per_lane.value, true>(f);
        };
        if (a.E <= kSub) values(std::integral_constant<int, 1>());
        else if (a.E <= 2 * kSub) values(std::integral_constant<int, 2>());
        else values(std::integral_constant<int, kShortValues>());
      } else {
        // granules at any alignment; the last one of a row that ends inside it is drawn back, and the values it shares with the one
        // before are left out
        const auto ask = [&](int g0, u32x4& x) { x = *reinterpret_cast<const u32x4_gate*>(row + min(g0 * V, a.E - V) * static_cast<int>(gb)); };
        const auto take = [&](int g0, u32x4 x, float* f) {
          const int j0 = min(g0 * V, a.E - V);
          each_value<GD>(x, [&](float val, int i) {
            const int j = j0 + i;
            f[i] = ((j >= g0 * V) & (j != e[0]) & (j != e[1])) ? val : -INFINITY;
          });
        };
        if (n <= kSub) {
          float f[V];
          u32x4 x;
          ask(sub, x);
          take(sub, x, f);
          ms.template add<V, true>(f);
        } else {
          for (int g0 = sub; g0 < n; g0 += 2 * kSub) {  // two in flight per lane
            float f[2 * V];
            u32x4 x0, x1;
            ask(g0, x0), ask(g0 + kSub, x1);
            take(g0, x0, f), take(g0 + kSub, x1, f + V);
            ms.add(f);
          }
        }
      }
      // merge the kSub lanes' (max, sum) pairs: they are neighbours in the wave
#pragma unroll
      for (int o = 1; o < kSub; o <<= 1) {
        const float ot = __shfl_xor(ms.top, o, kWave), os = __shfl_xor(ms.sum, o, kWave);
        const float nt = fmaxf(ms.top, ot);
        // a lane that saw no value holds (-inf, 0): its term is 0 whatever the other maximum is
        ms.sum = (ms.sum > 0.f ? ms.sum * expf(ms.top - nt) : 0.f) + (os > 0.f ? os * expf(ot - nt) : 0.f);
        ms.top = nt;
      }
      top = ms.top;
      if (e[0] >= 0) top = fmaxf(top, raw[0]);
      if (e[1] >= 0) top = fmaxf(top, raw[1]);
      rest = ms.sum > 0.f ? ms.sum * expf(ms.top - top) : 0.f;
      g[0] = e[0] >= 0 ? expf(raw[0] - top) : 0.f;   // exponentials for now, probabilities below
      g[1] = e[1] >= 0 ? expf(raw[1] - top) : 0.f;
      inv = 1.f / (rest + g[0] + g[1]);              // a row has at least one entry, and the largest one adds 1
      rest *= inv;
      g[0] *= inv;
      g[1] *= inv;
    }
    float d[2] = {0.f, 0.f};
    if (K == 1) {
      d[0] = dy[0];
    } else {
      const float sum = g[0] + g[1];
      if (sum >= 1.1920929e-07f) {
        const float r = 1.f / (sum * sum);
        d[0] = (dy[0] - dy[1]) * g[1] * r;
        d[1] = (dy[1] - dy[0]) * g[0] * r;
      } else {  // the clamped denominator is a constant
        d[0] = dy[0] / 1.1920929e-07f;
        d[1] = dy[1] / 1.1920929e-07f;
      }
      if (e[0] < 0) d[0] = 0.f;
      if (e[1] < 0) d[1] = 0.f;
    }
    if (sub == 0) {
      sh.i1[t] = e[0];
      sh.i2[t] = e[1];
      sh.top[t] = top;
      sh.inv[t] = inv;
      if (LOGITS) {  // 1 - p_1 = rest + p_2 and 1 - p_2 = rest + p_1: sums of positive terms
        sh.c1[t] = d[0] * (rest + g[1]) - g[1] * d[1];
        sh.c2[t] = d[1] * (rest + g[0]) - g[0] * d[0];
        sh.rest[t] = -(g[0] * d[0] + g[1] * d[1]);
      } else {
        sh.c1[t] = d[0];
        sh.c2[t] = d[1];
        sh.rest[t] = 0.f;
      }
    }
  }
  __syncthreads();
  // ---- the workgroup's block of the result, in memory order ---------------------------------------------------
  const int ntok = min(kGradTokens, a.S - first);
  const size_t base = static_cast<size_t>(first) * a.E;  // first element of the block
  const auto value = [&](int tk, int ex, float x) -> float {
    float c = sh.rest[tk];
    if (ex == sh.i1[tk]) c = sh.c1[tk];
    if (K == 2 && ex == sh.i2[tk]) c = sh.c2[tk];
    if (!LOGITS) return c;
    return expf(x - sh.top[tk]) * sh.inv[tk] * c;
  };
  const int n = ntok * a.E;
  const char* src = static_cast<const char*>(a.gate) + base * gb;
  char* dst = static_cast<char*>(a.out) + base * gb;
  int done = 0;
  if constexpr (BLOCK != kValues) {
    // (64 rows of any length are whole granules, so every workgroup's block starts on one)
    done = n / V * V;
    for (int q = tid * V; q < done; q += kTile * V) {
      const int tk = q / a.E, ex = q - tk * a.E;
      u32x4 x = {0u, 0u, 0u, 0u}, r;
      if (LOGITS) x = *reinterpret_cast<const u32x4*>(src + q * gb);
      float v[V];
      each_value<GD>(x, [&](float val, int i) { v[i] = val; });
      if constexpr (BLOCK == kGranules) {
#pragma unroll
        for (int i = 0; i < V; ++i) v[i] = value(tk, ex + i, v[i]);
      } else {
        int t = tk, e = ex;
#pragma unroll
        for (int i = 0; i < V; ++i) {
          v[i] = value(t, e, v[i]);
          e += 1;
          t += e == a.E;
          e = e == a.E ? 0 : e;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (GD == LANCET_F32) {
          r[i] = __float_as_uint(v[i]);
        } else {
          const uint32_t l = GD == LANCET_BF16 ? f32_to_bf16(v[2 * i]) : f32_to_f16(v[2 * i]);
          const uint32_t h = GD == LANCET_BF16 ? f32_to_bf16(v[2 * i + 1]) : f32_to_f16(v[2 * i + 1]);
          r[i] = (l & 0xffffu) | (h << 16);
        }
      }
      *reinterpret_cast<u32x4*>(dst + q * gb) = r;
    }
  }
  // what granules do not cover: everything, or the end of the last tokens
  for (int q = done + tid; q < n; q += kTile) {
    const int tk = q / a.E;
    const int ex = q - tk * a.E;
    const float x = LOGITS ? ld_gate(a.gate, base + q, GD) : 0.f;
    st_gate(a.out, base + q, value(tk, ex, x), GD);
  }
}

template <int K, int GD, bool LOGITS>
static void dgate_launch(const GateGradArgs& a, int block, hipStream_t st) {
  const int blocks = (a.S + kGradTokens - 1) / kGradTokens;
  if (block == kGranules) encode_dgate_kernel<K, GD, LOGITS, kGranules><<<blocks, kTile, 0, st>>>(a);
  else if (block == kCutGranules) encode_dgate_kernel<K, GD, LOGITS, kCutGranules><<<blocks, kTile, 0, st>>>(a);
  else encode_dgate_kernel<K, GD, LOGITS, kValues><<<blocks, kTile, 0, st>>>(a);
}

// Rows that end inside granules are written in granules from this length on (bytes): below, few threads have one, each with a chain
// of lookups.  Values / granules, us, 131072 top-2 on logits: 10 bf16 8.2 / 8.7, 12 bf16 8.4 / 8.8, 5 fp32 6.7 / 6.9; 14 fp32 9.7 / 9.4, and of 500
// tokens 3.6 / 3.3, 28 bf16 5.4 / 4.3.
constexpr int kCutRowBytes = 48;

hipError_t run_encode_dgate(const void* dy, const void* gate, const int32_t* idx, int S, int E, int K, bool is_logits,
                            int gate_dtype, void* out, hipStream_t st) {
  if (S == 0) return hipSuccess;
  GateGradArgs a;
  a.dy = dy;
  a.gate = gate;
  a.idx = idx;
  a.out = out;
  a.S = S;
  a.E = E;
  const int gb = gate_dtype == LANCET_F32 ? 4 : 2;
  const bool aligned = ((reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
  const bool whole_rows = static_cast<size_t>(E) * gb % 16 == 0;
  const int block = !aligned ? kValues : whole_rows ? kGranules : E * gb >= kCutRowBytes ? kCutGranules : kValues;
  LANCET_GATE_SWITCH(gate_dtype,
    if (K == 1) {
      if (is_logits) dgate_launch<1, GD, true>(a, block, st);
      else dgate_launch<1, GD, false>(a, block, st);
    } else {
      if (is_logits) dgate_launch<2, GD, true>(a, block, st);
      else dgate_launch<2, GD, false>(a, block, st);
    })
  return hipGetLastError();
}

}  // namespace lancet
