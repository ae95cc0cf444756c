// lbvh::builder<double> on gfx950 (lbvh.h:549-558 with scalar_type = double).
//
// The FP64 builder differs from builder<float> in three ways that change
// every byte of its output: codes are u64 (morton_domain<8> = 2^20 cells per
// axis, morton_encoder<8>), the arithmetic of centres, bounds and
// quantisation is FP64, and nodes are 64 bytes {aabb<double>, u64 left, u64
// right} with the leaf flag in bit 63.  The pipeline:
//   1. k_f64_bounds / k_f64_bounds_final: centroid bounds, std::min /
//      std::max semantics (lbvh.h:1282-1293, 1539-1543);
//   2. k_f64_encode: u64 codes (lbvh.h:1432-1473) and the digit histograms
//      of the radix passes the engine's sort reads (u64 keys, stable by
//      primitive id: one legal output of lbvh.h:1126-1134);
//   3. k_f64_tree_local / k_f64_tree_top: the tree and its boxes bottom up in
//      one pass, to the nodes of divide_node (lbvh.h:1588-1688, numbers
//      included) and union_of(left, right) (lbvh.h:1827-1866: box of the left
//      child, then the union with the right, left operand first); nodes
//      inside a workgroup's chunk of leaves finish in LDS, the few whose range
//      crosses a chunk boundary in a second kernel.
// The input is the converter's boxes (boxes48[i] = converter(primitives[i]),
// 6 doubles, 16-byte aligned).  Traffic is HBM-bound integer/FP64 work with
// no reuse beyond the sort, so the kernels stream with grid-stride loops.
#include "device_common.hpp"
#include "engine.hpp"

namespace lbvh_dev {

constexpr int kF64Block = 256;
constexpr uint32_t kF64BoundsBlocks = 1024;
constexpr uint32_t kF64EncodeBlocks = 512;
// Two encode workgroups a CU at 1M boxes (one per sort chunk) keep 16 waves
// with four boxes each in flight.
constexpr int kF64EncodeBlock = 512;
constexpr int kF64Unroll = 4;
constexpr uint64_t kLeafBit64 = 0x8000000000000000ull;

// libstdc++ std::min / std::max (the vector min/max behind union_of).
__device__ __forceinline__ double
std_min_d(double a, double b)
{
  return (b < a) ? b : a;
}
__device__ __forceinline__ double
std_max_d(double a, double b)
{
  return (a < b) ? b : a;
}

struct Box64
{
  double lo[3];
  double hi[3];
};

__device__ __forceinline__ Box64
load_box64(const double* __restrict__ boxes, uint64_t i)
{
  const double2* p = reinterpret_cast<const double2*>(boxes + 6 * i);
  double2 a = p[0], b = p[1], c = p[2];
  Box64 o;
  o.lo[0] = a.x;
  o.lo[1] = a.y;
  o.lo[2] = b.x;
  o.hi[0] = b.y;
  o.hi[1] = c.x;
  o.hi[2] = c.y;
  return o;
}

// center_of (lbvh.h:1164-1167): (min + max) * 0.5 per component.
__device__ __forceinline__ void
centre64(const Box64& b, double c[3])
{
#pragma unroll
  for (int k = 0; k < 3; k++)
    c[k] = (b.lo[k] + b.hi[k]) * 0.5;
}

// Workgroup-wide std::min / std::max of lo[3] / hi[3] into s[6]; accumulators
// start at +-inf and a NaN centre never replaces them, so the combination
// order does not change the result (signed zeros aside, which quantise alike).
__device__ __forceinline__ void
block_bounds(double lo[3], double hi[3], double* s_part)
{
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      lo[k] = std_min_d(lo[k], __shfl_xor(lo[k], off, kWave));
      hi[k] = std_max_d(hi[k], __shfl_xor(hi[k], off, kWave));
    }
  }
  const int wave = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      s_part[wave * 6 + k] = lo[k];
      s_part[wave * 6 + 3 + k] = hi[k];
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kF64Block / kWave; w++) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        s_part[k] = std_min_d(s_part[k], s_part[w * 6 + k]);
        s_part[3 + k] = std_max_d(s_part[3 + k], s_part[w * 6 + 3 + k]);
      }
    }
  }
  __syncthreads();
}

// Also clears zero[0 .. zero_words).
__global__ __launch_bounds__(kF64Block) void
k_f64_bounds(const double* __restrict__ boxes, uint64_t n, double* __restrict__ partials,
             uint32_t* __restrict__ zero, uint32_t zero_words)
{
  __shared__ double s_part[6 * (kF64Block / kWave)];
  double lo[3], hi[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    lo[k] = __builtin_inf();
    hi[k] = -__builtin_inf();
  }
  const uint64_t stride = uint64_t(gridDim.x) * kF64Block;
  for (uint64_t j = uint64_t(blockIdx.x) * kF64Block + threadIdx.x; j < zero_words; j += stride)
    zero[j] = 0u;
  for (uint64_t i0 = uint64_t(blockIdx.x) * kF64Block + threadIdx.x; i0 < n;
       i0 += stride * kF64Unroll) {
    // all loads in flight together (past the end: the last box again, which
    // changes no minimum or maximum)
    Box64 b[kF64Unroll];
#pragma unroll
    for (int u = 0; u < kF64Unroll; u++) {
      const uint64_t i = i0 + u * stride;
      b[u] = load_box64(boxes, i < n ? i : n - 1);
    }
#pragma unroll
    for (int u = 0; u < kF64Unroll; u++) {
      double c[3];
      centre64(b[u], c);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        lo[k] = std_min_d(lo[k], c[k]);
        hi[k] = std_max_d(hi[k], c[k]);
      }
    }
  }
  block_bounds(lo, hi, s_part);
  if (threadIdx.x < 6)
    partials[size_t(blockIdx.x) * 6 + threadIdx.x] = s_part[threadIdx.x];
}

// scale = 2^20 / (extent + 1) of every axis (lbvh.h:1432-1473).
__device__ __forceinline__ void
morton_scale64(const double* lo, const double* hi, double scale[3])
{
#pragma unroll
  for (int k = 0; k < 3; k++) {
    double ext = hi[k] - lo[k];
    scale[k] = 1048576.0 / (ext + 1.0);
  }
}

// The union of the partials to bounds[0 .. 6), and in the first word of
// bounds[6] the number of low bits that the codes use: the highest of the far
// corner's (no cell is beyond hi's), 61 to 63 when `extent + 1` rounds to the
// extent and hi falls into cell 2^20.
__global__ __launch_bounds__(kF64Block) void
k_f64_bounds_final(const double* __restrict__ partials, uint32_t nparts,
                   double* __restrict__ bounds)
{
  __shared__ double s_part[6 * (kF64Block / kWave)];
  double lo[3], hi[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    lo[k] = __builtin_inf();
    hi[k] = -__builtin_inf();
  }
  for (uint32_t p = threadIdx.x; p < nparts; p += kF64Block) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      lo[k] = std_min_d(lo[k], partials[size_t(p) * 6 + k]);
      hi[k] = std_max_d(hi[k], partials[size_t(p) * 6 + 3 + k]);
    }
  }
  block_bounds(lo, hi, s_part);
  if (threadIdx.x < 6)
    bounds[threadIdx.x] = s_part[threadIdx.x];
  if (threadIdx.x == 0) {
    double scale[3];
    morton_scale64(s_part, s_part + 3, scale);
    uint32_t used = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      double d = s_part[3 + k] - s_part[k];
      uint64_t q = uint64_t(d * scale[k]);
      q = q < 0x1fffffull ? q : 0x1fffffull; // what the expansion keeps
      const uint32_t u = q ? 3u * (64u - uint32_t(__clzll((long long)q))) - uint32_t(k) : 0u;
      used = u > used ? u : used;
    }
    *reinterpret_cast<uint32_t*>(bounds + 6) = used;
  }
}

// morton_encoder<8>::expand (lbvh.h:1377-1385): 20 bits to every third bit.
__device__ __forceinline__ uint64_t
expand20_d(uint64_t n)
{
  n = (n | n << 32) & 0x001f00000000ffffull;
  n = (n | n << 16) & 0x001f0000ff0000ffull;
  n = (n | n << 8) & 0x100f00f00f00f00full;
  n = (n | n << 4) & 0x10c30c30c30c30c3ull;
  n = (n | n << 2) & 0x1249249249249249ull;
  return n;
}

// Codes (lbvh.h:1432-1473 in FP64: scale = 2^20 / (extent + 1), q = (c -
// min) * scale truncated to u64) and the digit histograms of passes
// first_pass .. passes - 1, counted in LDS and added to hist[(p - first_pass)
// * radix + d] (zero before).  window: those passes' digits end at the highest
// code bit in use (bounds[6]) instead of starting at p * digit_bits.  counts != nullptr: workgroup g encodes the sort
// chunk [g * chunk, (g + 1) * chunk) and also writes its counts of pass
// first_pass to counts[d * gridDim.x + g], so the sort's first pass needs no
// count pass of its own.  1M boxes: 21 us and a count pass of 9-10 -> 17-19 us
// (a clearing launch of 2 us went to the bounds kernel).
__global__ __launch_bounds__(kF64EncodeBlock) void
k_f64_encode(const double* __restrict__ boxes, uint64_t n, const double* __restrict__ bounds,
             uint64_t* __restrict__ codes, uint32_t* __restrict__ hist, int digit_bits,
             int first_pass, int passes, bool window, uint32_t* __restrict__ counts,
             uint64_t chunk)
{
  extern __shared__ uint32_t s_hist[];
  const int radix = 1 << digit_bits;
  const int digits = passes - first_pass;
  const int words = radix * digits;
  for (int j = threadIdx.x; j < words; j += kF64EncodeBlock)
    s_hist[j] = 0u;
  double bmin[3], scale[3];
#pragma unroll
  for (int k = 0; k < 3; k++)
    bmin[k] = bounds[k];
  morton_scale64(bmin, bounds + 3, scale);
  int shift0 = first_pass * digit_bits;
  if (window) {
    const int used = int(*reinterpret_cast<const uint32_t*>(bounds + 6));
    shift0 = used > digits * digit_bits ? used - digits * digit_bits : 0;
  }
  __syncthreads();
  const uint64_t mask = uint64_t(radix - 1);
  uint64_t first = uint64_t(blockIdx.x) * kF64EncodeBlock + threadIdx.x;
  uint64_t limit = n;
  uint64_t stride = uint64_t(gridDim.x) * kF64EncodeBlock;
  if (counts) {
    const uint64_t b = uint64_t(blockIdx.x) * chunk;
    first = b + threadIdx.x;
    limit = b + chunk < n ? b + chunk : n;
    stride = kF64EncodeBlock;
  }
  for (uint64_t i0 = first; i0 < limit; i0 += stride * kF64Unroll) {
    Box64 b[kF64Unroll];
#pragma unroll
    for (int u = 0; u < kF64Unroll; u++) {
      const uint64_t i = i0 + u * stride;
      b[u] = load_box64(boxes, i < limit ? i : limit - 1);
    }
#pragma unroll
    for (int u = 0; u < kF64Unroll; u++) {
      const uint64_t i = i0 + u * stride;
      if (i >= limit)
        continue;
      double c[3];
      centre64(b[u], c);
      uint64_t q[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        double d = c[k] - bmin[k];
        q[k] = uint64_t(d * scale[k]);
      }
      const uint64_t code =
        (expand20_d(q[0]) << 2) | (expand20_d(q[1]) << 1) | expand20_d(q[2]);
      codes[i] = code;
      for (int p = 0; p < digits; p++)
        atomicAdd(&s_hist[p * radix + int((code >> (shift0 + p * digit_bits)) & mask)], 1u);
    }
  }
  __syncthreads();
  for (int j = threadIdx.x; j < words; j += kF64EncodeBlock) {
    const uint32_t v = s_hist[j];
    if (v)
      atomicAdd(&hist[j], v);
  }
  if (counts)
    for (int d = threadIdx.x; d < radix; d += kF64EncodeBlock)
      counts[size_t(d) * gridDim.x + blockIdx.x] = s_hist[d];
}

__device__ __forceinline__ Box64
box_union64(const Box64& l, const Box64& r)
{
  Box64 o;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    o.lo[k] = std_min_d(l.lo[k], r.lo[k]);
    o.hi[k] = std_max_d(l.hi[k], r.hi[k]);
  }
  return o;
}

__device__ __forceinline__ void
store_box64(double* p, const Box64& b)
{
  double2* q = reinterpret_cast<double2*>(p);
  q[0] = make_double2(b.lo[0], b.lo[1]);
  q[1] = make_double2(b.lo[2], b.hi[0]);
  q[2] = make_double2(b.hi[1], b.hi[2]);
}

// Leaves per tree workgroup (one thread each).
constexpr int kF64Leaves = 512;

// calc_delta (lbvh.h:1602-1621) of sorted positions k - 1 and k, plus one: the
// common leading bits of the codes, of the positions after them for equal
// codes, 0 beyond either end.  At most 128.
__device__ __forceinline__ uint8_t
delta_before(const uint64_t* __restrict__ codes, uint64_t n, uint64_t k)
{
  if (k == 0 || k >= n)
    return 0;
  const uint64_t a = codes[k - 1], b = codes[k];
  return uint8_t(a == b ? __clzll((long long)((k - 1) ^ k)) + 65
                        : __clzll((long long)(a ^ b)) + 1);
}

// The number of the node over positions [l, r], whose deltas to the outside
// are dl and dr (delta_before of l and of r + 1): the side of the larger one
// is where its sibling lies, and divide_node (lbvh.h:1588-1688) numbers a
// left child by its last position, a right child by its first and the root 0.
// The deltas around a node are different, but for the root's.
__device__ __forceinline__ uint32_t
node_number(uint32_t l, uint32_t r, uint32_t dl, uint32_t dr)
{
  return dl >= dr ? l : r;
}

// A node's 64-byte record; the children meet between positions g and g + 1.  A
// leaf names its sorted position, or (ids != nullptr) the primitive there.
__device__ __forceinline__ void
store_node64(uint64_t* __restrict__ node_words, uint32_t p, const Box64& b,
             const uint32_t* __restrict__ ids, uint32_t l, uint32_t g, uint32_t r)
{
  uint64_t left = g, right = uint64_t(g) + 1;
  if (l == g)
    left = (ids ? uint64_t(ids[g]) : left) | kLeafBit64;
  if (r == g + 1)
    right = (ids ? uint64_t(ids[g + 1]) : right) | kLeafBit64;
  uint64_t* q = node_words + size_t(p) * 8;
  store_box64(reinterpret_cast<double*>(q), b);
  *reinterpret_cast<ulonglong2*>(q + 6) = make_ulonglong2(left, right);
}

// Tree and boxes bottom up, part 1: one thread per sorted leaf position.  A
// node knows from the deltas on its two sides which one its parent's split g
// is on, and the two children of a split meet there: each leaves its box in
// LDS under its own number (a leaf's is its position; the internal node of
// that number holds this leaf, so it is made after the leaf's box was read)
// and exchanges the far end of its range with the split's flag; the second
// takes the union (left operand first, union_of of lbvh.h:1208-1213) and
// climbs on.  No search for ranges and splits and no parent links.
// What is left over (a child whose split is at the chunk's edge, or whose
// sibling reaches beyond it: then its flag is still set at the end) goes to
// the chunk's queue as {number, far end}, its box to `stage`.
// Bound by the climb (the deepest lane's steps, each LDS to LDS).  One box per
// number and not per child keeps it to 27 KB of LDS: four workgroups a CU.  1M
// boxes, this kernel + part 2: 58 + 53 us, where divide_node's searches, a
// flag clear and two fit kernels over parent links took 41 + 5 + 59 + 58; with
// 1,024 leaves a workgroup 64 + 52.
__global__ __launch_bounds__(kF64Leaves) void
k_f64_tree_local(const uint64_t* __restrict__ codes, const double* __restrict__ boxes, uint64_t n,
                 const uint32_t* __restrict__ ids, uint64_t* __restrict__ node_words,
                 uint8_t* __restrict__ deltas, uint32_t* __restrict__ flags,
                 double* __restrict__ stage, uint2* __restrict__ queue,
                 uint32_t* __restrict__ queue_count)
{
  __shared__ double s_box[6][kF64Leaves];
  __shared__ uint32_t s_flag[kF64Leaves];
  __shared__ uint8_t s_delta[kF64Leaves + 1];
  __shared__ uint32_t s_queued;
  const uint32_t first = uint32_t(blockIdx.x) * uint32_t(kF64Leaves);
  const uint32_t t = threadIdx.x;
  const uint32_t m = uint32_t(n - first < uint64_t(kF64Leaves) ? n - first : kF64Leaves);
  uint2* my_queue = queue + size_t(blockIdx.x) * kF64Leaves;
  const auto push = [&](uint32_t number, uint32_t far, const Box64& b) {
    if (number != far)
      store_box64(stage + size_t(first + number) * 6, b);
    my_queue[atomicAdd(&s_queued, 1u)] = make_uint2(first + number, first + far);
  };
  s_flag[t] = 0u;
  if (t == 0) {
    s_queued = 0u;
    s_delta[m] = delta_before(codes, n, uint64_t(first) + m);
    if (first + m == n)
      deltas[n] = 0;
  }
  Box64 box;
  if (t < m) {
    const uint32_t k = first + t;
    const uint8_t d = delta_before(codes, n, k);
    s_delta[t] = d;
    deltas[k] = d;
    flags[k] = 0u; // for part 2
    box = load_box64(boxes, ids ? ids[k] : k);
  }
  __syncthreads();
  if (t < m) {
    uint32_t l = t, r = t, dl = s_delta[t], dr = s_delta[t + 1];
    for (;;) {
      const bool right = dl > dr;
      const uint32_t number = right ? l : r, far = right ? r : l;
      if (right ? l == 0 : r + 1 == m) {
        push(number, far, box);
        break;
      }
      const uint32_t g = right ? l - 1 : r;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        s_box[c][number] = box.lo[c];
        s_box[3 + c][number] = box.hi[c];
      }
      const uint32_t met = __hip_atomic_exchange(&s_flag[g], far + 1, __ATOMIC_ACQ_REL,
                                                 __HIP_MEMORY_SCOPE_WORKGROUP);
      if (met == 0u)
        break;
      s_flag[g] = 0u;
      const uint32_t other = right ? g : g + 1;
      Box64 ob;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        ob.lo[c] = s_box[c][other];
        ob.hi[c] = s_box[3 + c][other];
      }
      if (right) {
        l = met - 1;
        dl = s_delta[l];
        box = box_union64(ob, box);
      } else {
        r = met - 1;
        dr = s_delta[r + 1];
        box = box_union64(box, ob);
      }
      store_node64(node_words, first + node_number(l, r, dl, dr), box, ids, first + l, first + g,
                   first + r);
      if (dl == dr) // the root
        break;
    }
  }
  __syncthreads();
  const uint32_t met = s_flag[t];
  if (met) {
    const uint32_t far = met - 1, number = far <= t ? t : t + 1;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      box.lo[c] = s_box[c][number];
      box.hi[c] = s_box[3 + c][number];
    }
    push(number, far, box);
  }
  __syncthreads();
  if (t == 0)
    queue_count[blockIdx.x] = s_queued;
}

// Part 2: the nodes whose range crosses a chunk boundary (all ancestors of
// such a node do too).  One wave per chunk takes the chunk's queued children;
// each climbs by exchanging far ends with a device-scope flag per split: the
// second arrival reads the sibling's box (input box for a leaf, `stage`
// otherwise), writes the node's record, publishes its box to `stage` with
// device-coherent stores and drains them before the next exchange.  flags[]
// is zero from part 1.  Bound by that chain (drain, exchange, load) a level;
// storing the record after the exchange instead takes nothing off it.
__global__ __launch_bounds__(kWave) void
k_f64_tree_top(const double* __restrict__ boxes, uint64_t n, const uint32_t* __restrict__ ids,
               uint64_t* __restrict__ node_words, const uint8_t* __restrict__ deltas,
               uint32_t* flags, uint64_t* stage, const uint2* __restrict__ queue,
               const uint32_t* __restrict__ queue_count)
{
  const uint32_t count = queue_count[blockIdx.x];
  const uint2* my_queue = queue + size_t(blockIdx.x) * kF64Leaves;
  for (uint32_t q = threadIdx.x; q < count; q += kWave) {
    const uint2 e = my_queue[q];
    uint32_t l = e.x < e.y ? e.x : e.y, r = e.x < e.y ? e.y : e.x;
    uint32_t dl = deltas[l], dr = deltas[size_t(r) + 1];
    Box64 box = l == r ? load_box64(boxes, ids ? ids[l] : l)
                       : load_box64(reinterpret_cast<const double*>(stage), e.x);
    for (;;) {
      const bool right = dl > dr;
      const uint32_t g = right ? l - 1 : r;
      const uint32_t other = right ? g : g + 1;
      vmem_drain();
      const uint32_t met = atomic_exch_agent(&flags[g], (right ? r : l) + 1);
      if (met == 0u)
        break;
      const uint32_t far = met - 1;
      const uint32_t d = deltas[right ? size_t(far) : size_t(far) + 1];
      Box64 ob;
      if (far == other) {
        ob = load_box64(boxes, ids ? ids[other] : other);
      } else {
        const uint64_t* st = stage + size_t(other) * 6;
#pragma unroll
        for (int c = 0; c < 3; c++) {
          ob.lo[c] = __longlong_as_double((long long)coherent_load_u64(st + c));
          ob.hi[c] = __longlong_as_double((long long)coherent_load_u64(st + 3 + c));
        }
      }
      if (right) {
        l = far;
        dl = d;
        box = box_union64(ob, box);
      } else {
        r = far;
        dr = d;
        box = box_union64(box, ob);
      }
      const uint32_t p = node_number(l, r, dl, dr);
      store_node64(node_words, p, box, ids, l, g, r);
      if (dl == dr) // the root
        break;
      uint64_t* st = stage + size_t(p) * 6;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        coherent_store_u64(st + c, (uint64_t)__double_as_longlong(box.lo[c]));
        coherent_store_u64(st + 3 + c, (uint64_t)__double_as_longlong(box.hi[c]));
      }
    }
  }
}

} // namespace lbvh_dev

namespace lbvh_eng {

using namespace lbvh_dev;

uint32_t
f64_bounds_blocks(uint64_t n)
{
  uint64_t b = (n + kF64Block * kF64Unroll - 1) / (kF64Block * kF64Unroll);
  return uint32_t(b < kF64BoundsBlocks ? (b ? b : 1) : kF64BoundsBlocks);
}

hipError_t
launch_f64_bounds(const double* boxes, uint64_t n, double* partials, double* bounds,
                  uint32_t* zero, uint32_t zero_words, hipStream_t s)
{
  const uint32_t g = f64_bounds_blocks(n);
  hipLaunchKernelGGL(k_f64_bounds, dim3(g), dim3(kF64Block), 0, s, boxes, n, partials, zero,
                     zero_words);
  hipLaunchKernelGGL(k_f64_bounds_final, dim3(1), dim3(kF64Block), 0, s,
                     static_cast<const double*>(partials), g, bounds);
  return hipGetLastError();
}

hipError_t
launch_f64_encode(const double* boxes, uint64_t n, const double* bounds, uint64_t* codes,
                  uint32_t* hist, int digit_bits, int first_pass, int passes, bool window,
                  uint32_t* counts, uint32_t chunks, uint64_t chunk, hipStream_t s)
{
  const size_t lds = (size_t(4) << digit_bits) * size_t(passes - first_pass);
  if (first_pass < 0 || first_pass > passes || lds > 64 * 1024 ||
      (counts && (!chunks || uint64_t(chunks) * chunk < n)))
    return hipErrorInvalidValue;
  // without chunks few workgroups: each flushes up to passes x radix histogram words
  uint64_t b = (n + kF64EncodeBlock * kF64Unroll - 1) / (kF64EncodeBlock * kF64Unroll);
  const uint32_t g = counts ? chunks : uint32_t(b < kF64EncodeBlocks ? b : kF64EncodeBlocks);
  // the kernel counts pass p at (p - first_pass) * radix of its pointer
  hipLaunchKernelGGL(k_f64_encode, dim3(g), dim3(kF64EncodeBlock), lds, s, boxes, n, bounds,
                     codes, hist + size_t(first_pass) * (size_t(1) << digit_bits), digit_bits,
                     first_pass, passes, window, counts, chunk);
  return hipGetLastError();
}

// Scratch of the FP64 tree, in order: fit queues [chunks * kF64Leaves] (8
// bytes an entry), fit flags [n], queue counts [chunks] (u32), deltas [n + 1]
// (u8), then 16-byte aligned staging boxes [n - 1] of 48 bytes.
struct F64Scratch
{
  uint2* queue;
  uint32_t *flags, *count;
  uint8_t* deltas;
  double* stage;
};

static uint64_t
f64_chunks(uint64_t n)
{
  return (n + kF64Leaves - 1) / kF64Leaves;
}

static uint64_t
f64_stage_offset(uint64_t n)
{
  const uint64_t b = f64_chunks(n) * (8 * kF64Leaves + 4) + 4 * n + (n + 1);
  return (b + 15) & ~uint64_t(15);
}

static F64Scratch
f64_scratch(void* base, uint64_t n)
{
  F64Scratch f;
  f.queue = static_cast<uint2*>(base);
  f.flags = reinterpret_cast<uint32_t*>(f.queue + f64_chunks(n) * kF64Leaves);
  f.count = f.flags + n;
  f.deltas = reinterpret_cast<uint8_t*>(f.count + f64_chunks(n));
  f.stage = reinterpret_cast<double*>(static_cast<char*>(base) + f64_stage_offset(n));
  return f;
}

uint64_t
f64_tree_scratch_bytes(uint64_t n)
{
  return f64_stage_offset(n) + 48 * (n - 1);
}

hipError_t
launch_f64_tree(const uint64_t* sorted, const uint32_t* ids, const double* boxes, uint64_t n,
                void* nodes, void* scratch, hipStream_t s)
{
  if (n < 2 || n > 0x7fffffffull)
    return hipErrorInvalidValue;
  uint64_t* w = static_cast<uint64_t*>(nodes);
  const F64Scratch f = f64_scratch(scratch, n);
  const uint32_t chunks = uint32_t(f64_chunks(n));
  hipLaunchKernelGGL(k_f64_tree_local, dim3(chunks), dim3(kF64Leaves), 0, s, sorted, boxes, n, ids,
                     w, f.deltas, f.flags, f.stage, f.queue, f.count);
  if (chunks > 1) // else the one workgroup made the root
    hipLaunchKernelGGL(k_f64_tree_top, dim3(chunks), dim3(kWave), 0, s, boxes, n, ids, w,
                       static_cast<const uint8_t*>(f.deltas), f.flags,
                       reinterpret_cast<uint64_t*>(f.stage), static_cast<const uint2*>(f.queue),
                       static_cast<const uint32_t*>(f.count));
  return hipGetLastError();
}

} // namespace lbvh_eng
