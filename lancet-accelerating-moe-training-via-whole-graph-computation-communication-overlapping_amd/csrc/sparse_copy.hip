// Copies between a 3-D "sparse" buffer, in which block b along one axis holds only its first n_b
// elements, and the packed stream of those elements (memcpy_sparse_to_cont_3d /
// memcpy_cont_to_sparse_3d, src/op/dialect/cuda/kernels/sparse_memcpy.cu:11-96).  n_b comes from a
// device array of uint64 element counts read with a stride and an offset, which is how a caller
// picks one column of elements_per_expert viewed as [G, LE].
//
//   n_b   = counts[b*stride + offset] * scale / shrink
//   off_b = (sum_{j<b} counts[j*stride + offset]) * scale / shrink          (sum first, as the source does)
//   axis 0: stream[off_b + t] <-> buf[b, t / dim2, t % dim2]
//   axis 1: stream[off_b + t] <-> buf[t / dim2, b, t % dim2]
// With a second array `starts` (same indexing and scaling as the counts) block b's elements are
// [start_b, start_b + n_b) instead of [0, n_b): the rows one token partition owns inside a buffer that
// several partitions share.
//
// The grid is (chunks, blocks along the axis): unlike one workgroup per block, a few long blocks
// still fill the chip.  Elements move in 16-byte granules where offsets and rows allow it.
#include "common.hpp"
#include "launchers.hpp"

namespace lancet {

namespace {

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const uint32_t lo = __shfl_xor(static_cast<uint32_t>(v), o, kWave);
    const uint32_t hi = __shfl_xor(static_cast<uint32_t>(v >> 32), o, kWave);
    v += (static_cast<uint64_t>(hi) << 32) | lo;
  }
  return v;
}

// position of stream element t of block b inside the 3-D buffer
template <int AXIS>
__device__ __forceinline__ size_t sparse_index(uint32_t b, uint32_t t, uint32_t dim1, uint32_t dim2) {
  if (AXIS == 0) return static_cast<size_t>(b) * dim1 * dim2 + t;
  const uint32_t r = t / dim2;
  return (static_cast<size_t>(r) * dim1 + b) * dim2 + (t - r * dim2);
}

// Granules per thread and tile: the tile of a workgroup is kTile * kCopyBatch of them, one behind the other, all loads
// of a thread in flight before its first store (pipeline as below: one / two / four 1406 / 1349 / 1336 us).
constexpr uint32_t kCopyBatch = 4;

// 16 bytes.  Aligned ones: non-temporal loads (nobody reads the source again) and plain stores: what a copy writes is the
// next copy's or the decode's input and stays in the cache for it (four-partition pipeline of 65536 x 4096 bf16 top-2:
// 1467 us with non-temporal stores, 1336 with plain ones; plain loads as well 1478).  Where they are not aligned (the
// hardware takes them at any element) they share lines with their neighbours and both are plain.
typedef u32x4 u32x4_any __attribute__((aligned(2)));
template <bool ALIGNED>
__device__ __forceinline__ u32x4 ld_granule(const void* p) {
  if (ALIGNED) return ld_stream(static_cast<const u32x4*>(p));
  return *static_cast<const u32x4_any*>(p);
}
template <bool ALIGNED>
__device__ __forceinline__ void st_granule(void* p, u32x4 x) {
  if (ALIGNED) *static_cast<u32x4*>(p) = x;
  else *static_cast<u32x4_any*>(p) = x;
}

// One block's elements [0, n) copied and, in buffer direction, [n, end) cleared; `in` / `out` are indexed by `at(t)` on the
// buffer's side and by t on the stream's.
template <typename EL, bool TO_CONT, bool ALIGNED, typename At>
__device__ __forceinline__ void copy_granules(const EL* in, EL* out, uint32_t n, uint32_t end, At at) {
  constexpr uint32_t kPer = 16 / sizeof(EL);
  const u32x4 zero = {0u, 0u, 0u, 0u};
  const uint32_t whole = n / kPer, end_vec = end / kPer;
  for (uint32_t base = blockIdx.x * (kTile * kCopyBatch); base < end_vec; base += gridDim.x * (kTile * kCopyBatch)) {
    const uint32_t v0 = base + threadIdx.x;
    u32x4 x[kCopyBatch];
    size_t place[kCopyBatch];
#pragma unroll
    for (uint32_t j = 0; j < kCopyBatch; ++j) {
      const uint32_t v = v0 + j * kTile;
      x[j] = zero;
      if (v < end_vec) place[j] = at(v * kPer);
      if (v < whole) x[j] = ld_granule<ALIGNED>(in + (TO_CONT ? place[j] : static_cast<size_t>(v) * kPer));
    }
#pragma unroll
    for (uint32_t j = 0; j < kCopyBatch; ++j) {
      const uint32_t v = v0 + j * kTile;
      if (v >= end_vec) continue;
      EL* to = out + (TO_CONT ? static_cast<size_t>(v) * kPer : place[j]);
      if (v != whole || n % kPer == 0) {
        st_granule<ALIGNED>(to, x[j]);
      } else {  // the granule that holds element n (in buffer direction with a fill behind it)
        for (uint32_t i = 0; i < kPer; ++i) to[i] = v * kPer + i < n ? in[static_cast<size_t>(v) * kPer + i] : EL(0);
      }
    }
  }
  const uint32_t t = end_vec * kPer + threadIdx.x;  // what is left of less than a granule
  if (blockIdx.x == 0 && t < end) {
    const size_t p = at(t);
    if (TO_CONT) out[t] = in[p];
    else out[p] = t < n ? in[t] : EL(0);
  }
}

// EL: element storage type.  TO_CONT: buffer -> stream, else stream -> buffer.  VEC: granules do not cross a run of the
// buffer (axis 0: one run per block; axis 1: rows of whole granules, the range's own start is checked here).  ALIGNED:
// the base pointers and the runs are aligned to granules.  ZERO_TAIL (only stream -> buffer): elements [n_b, block_cap) of
// every block are cleared.
// Bound by memory latency, so every wave asks for its block's counts at once, adds them up by itself and then has four
// granules in flight: 67M bf16 elements in 32 blocks, buffer to stream 53 us (5.1 TB/s) with one granule per thread behind
// a workgroup-wide sum, 43.6 (6.2 TB/s) now; stream to buffer 52 and 43.5 us.
template <typename EL, int AXIS, bool TO_CONT, bool VEC, bool ALIGNED, bool ZERO_TAIL>
__global__ __launch_bounds__(kTile) void sparse_copy_3d_kernel(const EL* __restrict__ src, EL* __restrict__ dst,
                                                               const uint64_t* __restrict__ counts,
                                                               const uint64_t* __restrict__ starts, int stride,
                                                               int offset, uint32_t dim1, uint32_t dim2,
                                                               uint32_t block_cap, uint64_t cont_cap, uint64_t scale,
                                                               uint64_t shrink) {
  const uint32_t b = blockIdx.y;
  const auto scaled = [&](uint64_t x) { return shrink == 1 ? x * scale : x * scale / shrink; };
  uint64_t acc = 0;
  for (uint32_t j = lane_id(); j < b; j += kWave) acc += counts[static_cast<size_t>(j) * stride + offset];
  uint64_t n64 = scaled(counts[static_cast<size_t>(b) * stride + offset]);
  uint64_t start64 = starts ? scaled(starts[static_cast<size_t>(b) * stride + offset]) : 0;
  // never leave the block or the stream
  if (start64 > block_cap) start64 = block_cap;
  if (n64 > block_cap - start64) n64 = block_cap - start64;
  const uint32_t start = static_cast<uint32_t>(start64);
  constexpr uint32_t kPer = 16 / sizeof(EL);
  const bool granules = VEC && (AXIS == 0 || start % kPer == 0);
  {
    const uint64_t most = (!TO_CONT && ZERO_TAIL) ? block_cap - start64 : n64;
    if (static_cast<uint64_t>(blockIdx.x) * kTile * (granules ? kCopyBatch * kPer : 1u) >= most) return;
  }
  const uint64_t off = scaled(wave_sum_u64(acc));
  if (off >= cont_cap) n64 = 0;
  else if (n64 > cont_cap - off) n64 = cont_cap - off;
  const uint32_t n = static_cast<uint32_t>(n64);
  const uint32_t end = (!TO_CONT && ZERO_TAIL) ? block_cap - start : n;  // the fill covers [start + n, block_cap)

  const auto at = [&](uint32_t t) { return sparse_index<AXIS>(b, start + t, dim1, dim2); };
  if (granules) {
    const EL* in = TO_CONT ? src : src + off;
    EL* out = TO_CONT ? dst + off : dst;
    if (ALIGNED && off % kPer == 0 && start % kPer == 0) copy_granules<EL, TO_CONT, true>(in, out, n, end, at);
    else copy_granules<EL, TO_CONT, false>(in, out, n, end, at);
    return;
  }
  for (uint32_t t = blockIdx.x * kTile + threadIdx.x; t < end; t += gridDim.x * kTile) {
    const size_t si = at(t);
    if (TO_CONT) dst[off + t] = src[si];
    else dst[si] = t < n ? src[off + t] : EL(0);
  }
}

template <typename EL, int AXIS, bool TO_CONT>
hipError_t launch(const void* src, void* dst, const uint64_t* counts, const uint64_t* starts, int stride, int offset, int nblocks, uint32_t dim1,
                  uint32_t dim2, uint32_t block_cap, uint64_t cont_cap, uint64_t scale, uint64_t shrink, bool vec, bool aligned,
                  bool zero_tail, hipStream_t st) {
  constexpr uint32_t kPer = 16 / sizeof(EL);
  const uint32_t per_wg = kTile * kPer * kCopyBatch;
  uint32_t chunks = (block_cap + per_wg - 1) / per_wg;
  if (chunks < 1) chunks = 1;
  if (chunks > 1024) chunks = 1024;
  const dim3 grid(chunks, static_cast<unsigned>(nblocks));
  const EL* s = static_cast<const EL*>(src);
  EL* d = static_cast<EL*>(dst);
#define LANCET_SPARSE_LAUNCH(V, A, Z) \
  sparse_copy_3d_kernel<EL, AXIS, TO_CONT, V, A, Z><<<grid, kTile, 0, st>>>(s, d, counts, starts, stride, offset, dim1, dim2, block_cap, cont_cap, scale, shrink)
#define LANCET_SPARSE_ROUTE(Z)                        \
  if (vec && aligned) LANCET_SPARSE_LAUNCH(true, true, Z); \
  else if (vec) LANCET_SPARSE_LAUNCH(true, false, Z); \
  else LANCET_SPARSE_LAUNCH(false, false, Z);
  if (!TO_CONT && zero_tail) {
    LANCET_SPARSE_ROUTE(true)
  } else {
    LANCET_SPARSE_ROUTE(false)
  }
#undef LANCET_SPARSE_ROUTE
#undef LANCET_SPARSE_LAUNCH
  return hipGetLastError();
}

template <typename EL>
hipError_t launch_el(const void* src, void* dst, const uint64_t* counts, const uint64_t* starts, int stride, int offset, int axis, int dim0,
                     int dim1, int dim2, uint64_t cont_cap, uint64_t scale, uint64_t shrink, bool to_cont,
                     bool zero_tail, hipStream_t st) {
  constexpr uint32_t kPer = 16 / sizeof(EL);
  const int nblocks = axis == 0 ? dim0 : dim1;
  const uint32_t block_cap = static_cast<uint32_t>(axis == 0 ? static_cast<int64_t>(dim1) * dim2 : static_cast<int64_t>(dim0) * dim2);
  if (nblocks == 0 || block_cap == 0) return hipSuccess;
  // axis 0 moves flat runs of dim1*dim2 elements, axis 1 runs of dim2
  const uint32_t run = axis == 0 ? block_cap : static_cast<uint32_t>(dim2);
  const bool vec = axis == 0 || run % kPer == 0;
  const bool aligned = run % kPer == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
  const uint32_t d1 = static_cast<uint32_t>(dim1), d2 = static_cast<uint32_t>(dim2);
  if (axis == 0) {
    return to_cont ? launch<EL, 0, true>(src, dst, counts, starts, stride, offset, nblocks, d1, d2, block_cap, cont_cap, scale, shrink, vec, aligned, zero_tail, st)
                   : launch<EL, 0, false>(src, dst, counts, starts, stride, offset, nblocks, d1, d2, block_cap, cont_cap, scale, shrink, vec, aligned, zero_tail, st);
  }
  return to_cont ? launch<EL, 1, true>(src, dst, counts, starts, stride, offset, nblocks, d1, d2, block_cap, cont_cap, scale, shrink, vec, aligned, zero_tail, st)
                 : launch<EL, 1, false>(src, dst, counts, starts, stride, offset, nblocks, d1, d2, block_cap, cont_cap, scale, shrink, vec, aligned, zero_tail, st);
}

}  // namespace

hipError_t run_sparse_copy_3d(const void* src, void* dst, const uint64_t* counts, const uint64_t* starts, int stride, int offset, int axis,
                              int dim0, int dim1, int dim2, uint64_t cont_cap, uint64_t scale, uint64_t shrink,
                              bool to_cont, bool zero_tail, int elem_bytes, hipStream_t st) {
  if (elem_bytes == 4)
    return launch_el<uint32_t>(src, dst, counts, starts, stride, offset, axis, dim0, dim1, dim2, cont_cap, scale, shrink, to_cont, zero_tail, st);
  return launch_el<uint16_t>(src, dst, counts, starts, stride, offset, axis, dim0, dim1, dim2, cont_cap, scale, shrink, to_cont, zero_tail, st);
}

}  // namespace lancet
