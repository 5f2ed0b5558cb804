// Arguments of the routing kernels, and what a token of a top-1 / top-2 encode becomes once its ranks and the totals are known
// (moe_route.hip, moe_encode_short.hip).
#pragma once
#include "select.hpp"

namespace lancet {

struct RouteArgs {
  const void* gate;       // [S,E] of gate_dtype (NULL when idx_in is given)
  const void* noise;      // [S,E] of gate_dtype or NULL: added for the second choice (K = 2)
  const int32_t* idx_in;  // launcher-level entry: expert per token already chosen (may alias idx_out)
  const int32_t* used_in; // [E] or NULL (= zeros)
  void* gates_s;          // [K*S] of gate_dtype (NULL when idx_in is given)
  int32_t* idx_out;       // [K*S]
  int32_t* loc_out;       // [K*S]
  int32_t* used_out;      // [E]
  uint64_t* elems_out;    // [E]
  ScanWs ws;
  int S, E, C, M;
  int ntiles;
  int is_logits;
  int gate_dtype;         // LANCET_F32 / _BF16 / _F16: storage type of gate, noise and gates_s
  int seg_rows;           // place kernel: tiles per segment of the segment sums, 0 = there are none
};

// Slots of a top-2 token: r1 / r2 = tokens before it with the same first / second choice, total1 = first choices of e2 in the
// batch.  Slot 1 is an ordinary top-1 encode; slot 2 a top-1 encode whose used capacity is slot 1's result; locations are in the
// merged layout (slot-2 rows follow slot-1 rows of the same expert).
struct Top2Place {
  int e1, l1, e2, l2;
};
__device__ __forceinline__ Top2Place place_top2(int e1, int r1, int e2, int r2, int u1, int u2, uint32_t total1, int E, int C) {
  const bool in1 = e1 >= 0 && e1 < E, in2 = e2 >= 0 && e2 < E;
  const bool keep1 = in1 && r1 < C - u1;
  const int64_t after1 = min(static_cast<int64_t>(u2) + (in2 ? total1 : 0u), static_cast<int64_t>(C));
  const bool keep2 = in2 && r2 < C - after1;
  return {keep1 ? e1 : -1, keep1 ? r1 : -1, keep2 ? e2 : -1, keep2 ? r2 + static_cast<int>(after1 - u2) : -1};
}

// route_count_kernel (moe_route.hip): selection, ranks inside the tiles and the tiles' counts, what the kernels that finish the
// routing start from
hipError_t run_route_count(const RouteArgs& a, int K, hipStream_t st);

}  // namespace lancet
