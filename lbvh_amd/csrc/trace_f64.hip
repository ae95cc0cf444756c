// Closest-hit traversal of builder<double> trees on gfx950.
//
// traverser<double> (lbvh.h:1874-1942) over node<double> records with
// triangle_intersector<double> (lbvh.h:2055-2075), in FP64 throughout:
// make_accel_ray (lbvh.h:991-1010) and the octant box test (lbvh.h:1071-1091,
// hit iff tmax >= max(0, tmin), lbvh.h:1023-1026) on the children's own
// boxes; the root pushed with tmin = +inf; a popped entry skipped when the
// closest hit so far is nearer than its tmin; leaf children intersected at
// once, left then right; hit children pushed far first, near last; a
// 128-entry stack that drops pushes when full (traversal_stack<double,128>,
// lbvh.h:1746-1789).  A leaf value names the triangle<double> record it tests
// (lbvh.h:1904-1905, 1915-1916) and the hit reports that value, u64 with
// UINT64_MAX for a miss (intersection_container<double>, lbvh.h:364-366).
#include "device_common.hpp"
#include "engine.hpp"

namespace lbvh_dev {

// lbvh::node<double> (lbvh.h:220-255): box {min xyz, max xyz}, left, right;
// bit 63 of left / right marks a leaf.
struct alignas(64) Node64
{
  double bmin[3];
  double bmax[3];
  uint64_t left;
  uint64_t right;
};
static_assert(sizeof(Node64) == 64, "node<double> is 64 bytes");

constexpr uint64_t kLeafBit64 = uint64_t(1) << 63;
// Two waves per workgroup: the 1M primary launch 1.10 ms with four, 1.00 ms
// with two (one timed the same).
constexpr int kTraceF64Block = 128;
constexpr int kStackF64 = 128;
// Stack entries kept in LDS per thread (a power of two, a ring; 16 KB per
// 128-thread workgroup).
constexpr int kStackF64Lds = 8;
// s_waitcnt operand: no vector memory operation outstanding (vmcnt 0, other
// counters at their maximum).
constexpr int kWaitVmem0F64 = 0x0F70;

__device__ __forceinline__ double
dm_min(double a, double b)
{
  return (a < b) ? a : b;
}
__device__ __forceinline__ double
dm_max(double a, double b)
{
  return (a > b) ? a : b;
}

// lbvh::math::dot (lbvh.h:621-630): accumulation starts from 0.
__device__ __forceinline__ double
ddot3(const double* a, const double* b)
{
  double out = 0.0;
  double px = a[0] * b[0];
  out = out + px;
  double py = a[1] * b[1];
  out = out + py;
  double pz = a[2] * b[2];
  out = out + pz;
  return out;
}

// lbvh::math::cross (lbvh.h:609-616)
__device__ __forceinline__ void
dcross3(const double* a, const double* b, double* o)
{
  double ay_bz = a[1] * b[2], az_by = a[2] * b[1];
  double az_bx = a[2] * b[0], ax_bz = a[0] * b[2];
  double ax_by = a[0] * b[1], ay_bx = a[1] * b[0];
  o[0] = ay_bz - az_by;
  o[1] = az_bx - ax_bz;
  o[2] = ax_by - ay_bx;
}

// The closest hit so far.
struct Hit64
{
  uint64_t prim = ~uint64_t(0);
  double t = INFINITY, u = 0.0, v = 0.0;
};

// triangle_intersector<double> on a triangle<double> record {p0, e0, e1,
// normal} (12 doubles) already loaded as six double2; a hit that beats the
// closest so far replaces it.
template<int MODE>
__device__ __forceinline__ void
isect_f64(const double2 (&q)[6], uint64_t id, const double o[3], const double d[3], double tmin,
          double tmax, Hit64& h)
{
  const double2 a = q[0], b = q[1], c = q[2], e = q[3], f = q[4], g = q[5];
  const double p0[3] = { a.x, a.y, b.x };
  const double e0[3] = { b.y, c.x, c.y };
  const double e1[3] = { e.x, e.y, f.x };
  const double nrm[3] = { f.y, g.x, g.y };
  double cc[3] = { p0[0] - o[0], p0[1] - o[1], p0[2] - o[2] };
  double r[3];
  dcross3(d, cc, r);
  double inv_det = 1.0 / ddot3(nrm, d);
  double u = ddot3(r, e1) * inv_det;
  double v = ddot3(r, e0) * inv_det;
  double w = (1.0 - u) - v;
  if ((u >= 0.0) && (v >= 0.0) && (w >= 0.0)) {
    double t = ddot3(nrm, cc) * inv_det;
    const bool take = (MODE == 0) ? (t < h.t) : ((t < h.t) || (t == h.t && id < h.prim));
    if ((t >= tmin) && (t <= tmax) && take) {
      h.prim = id;
      h.t = t;
      h.u = u;
      h.v = v;
    }
  }
}

// MODE 0: the first hit found wins ties (the reference's strict <);
// MODE 1: equal distances go to the lowest primitive value.
//
// Bound by instruction issue and by each visit's dependent fetch, as the FP32
// traversal, and built like it: no branch around loads, box tests or
// addresses, pruned entries dropped in a loop of their own, an LDS ring for
// the stack's top.  2,073,600 primary rays on the clustered 1M tree: 988 us
// with branches per child and a trip per pruned entry, 815 us so at three
// waves per SIMD (130 registers), 799 us held to the 128 registers of four
// (a ring of 4 entries: 823 us).
template<int MODE>
__global__ __launch_bounds__(kTraceF64Block, 4) void
k_trace_f64(const Node64* __restrict__ nodes, const double* __restrict__ tris, uint64_t n,
            const double* __restrict__ rays, uint64_t nrays, uint64_t* __restrict__ prim_out,
            double* __restrict__ t_out, double* __restrict__ uv_out)
{
  const uint64_t i = uint64_t(blockIdx.x) * kTraceF64Block + threadIdx.x;
  if (i >= nrays)
    return;
  const double2* rp = reinterpret_cast<const double2*>(rays + 8 * i);
  const double2 r0 = rp[0], r1 = rp[1], r2 = rp[2], r3 = rp[3];
  const double o[3] = { r0.x, r0.y, r1.x };
  const double d[3] = { r1.y, r2.x, r2.y };
  const double rtmin = r3.x, rtmax = r3.y;
  // make_accel_ray: rcp = 1 / dir, inv_pos = (-pos) * rcp, octant by sign
  double rcp[3], ipos[3];
  bool pos_dir[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    rcp[k] = 1.0 / d[k];
    double np = -o[k];
    ipos[k] = np * rcp[k];
    pos_dir[k] = d[k] > 0.0;
  }
  // The stack: capacity 128 (pushes onto a full stack are dropped).  An
  // entry stands for a pushed node and holds what its own record gave when
  // its box was tested: its two children (packed to 32 bits, bit 31 marking a
  // leaf, as every index is below 2^31) and the box's entry distance (the
  // reference's tmin), so popping it needs no further load.  The top entry
  // is kept in registers: a pop leaves it stale (the top is still entry
  // sp - 1), and its reload is issued after the children's fetches, so the
  // latencies overlap.  Of the entries below it the kStackF64Lds nearest the
  // top are in an LDS ring, one column per thread, the first `low` in a
  // private array.
  __shared__ uint2 s_lr[kStackF64Lds * kTraceF64Block];
  __shared__ double s_tmin[kStackF64Lds * kTraceF64Block];
  uint2 spill_lr[kStackF64];
  double spill_t[kStackF64];
  auto slot = [&](uint32_t e) { return (e & (kStackF64Lds - 1)) * kTraceF64Block + threadIdx.x; };
  auto pack = [](uint64_t v) -> uint32_t {
    return (v & kLeafBit64) ? (uint32_t(v) | 0x80000000u) : uint32_t(v);
  };
  uint2 top_lr = make_uint2(0u, 0u);
  double top_t = 0.0;
  uint32_t sp = 0, low = 0;
  bool stale = false;
  auto push = [&](uint2 lr, double tm) {
    if (sp > 0 && !stale) {
      const uint32_t e = sp - 1;
      if (e - low == uint32_t(kStackF64Lds)) {
        spill_lr[low] = s_lr[slot(low)];
        spill_t[low] = s_tmin[slot(low)];
        low++;
      }
      s_lr[slot(e)] = top_lr;
      s_tmin[slot(e)] = top_t;
    }
    stale = false;
    top_lr = lr;
    top_t = tm;
    sp++;
  };
  auto reload = [&]() { // a stale top (sp > 0)
    const uint32_t e = sp - 1;
    if (e < low) {
      top_lr = spill_lr[e];
      top_t = spill_t[e];
      low = e;
      // waited for here: left pending, it would make every later wait for a
      // child's data wait for more than that data
      __builtin_amdgcn_s_waitcnt(kWaitVmem0F64);
    } else {
      top_lr = s_lr[slot(e)];
      top_t = s_tmin[slot(e)];
    }
    stale = false;
  };
  Hit64 best;
  // The root is pushed and popped at once: its record gives the first two
  // children.  A child that would be pushed and popped again straight away
  // (the near one of two, or a single hit child) is taken directly, when its
  // push would have found room, so the visit order and the drop-when-full
  // rule are the reference's.
  if (n >= 2) {
    const ulonglong2 root = *reinterpret_cast<const ulonglong2*>(&nodes[0].left);
    uint32_t ch[2] = { pack(root.x), pack(root.y) };
    const char* const node_base = reinterpret_cast<const char*>(nodes);
    const char* const tri_base = reinterpret_cast<const char*>(tris);
    const uint32_t last_leaf = uint32_t(n) - 1u, last_node = uint32_t(n) - 2u;
    // A tree's traversal visits each of its n - 1 internal nodes at most
    // once; a caller's node array that is not a tree (a child cycle) ends
    // after n visits.
    for (uint32_t visits = 0; visits < n; visits++) {
      // both children's data at once: a leaf's triangle<double> record (96
      // bytes), an internal node's record (64); a child out of range (only
      // possible for a corrupt node array) is skipped, its loads go to the
      // array's last entry
      bool leaf[2], ok[2];
      uint32_t idx[2];
      const double2* at[2];
      double2 q[2][6];
#pragma unroll
      for (int side = 0; side < 2; side++) {
        leaf[side] = int32_t(ch[side]) < 0;
        const uint32_t x = ch[side] & 0x7fffffffu;
        const uint32_t lim = leaf[side] ? last_leaf : last_node;
        ok[side] = x <= lim;
        idx[side] = x < lim ? x : lim;
        const uint32_t more = leaf[side] ? idx[side] : 0u;
        const char* base = leaf[side] ? tri_base : node_base;
        at[side] = reinterpret_cast<const double2*>(base + (uint64_t(idx[side]) << 6) +
                                                    (uint64_t(more) << 5));
      }
#pragma unroll
      for (int side = 0; side < 2; side++) {
#pragma unroll
        for (int k = 0; k < 4; k++)
          q[side][k] = at[side][k];
        if (leaf[side]) {
          q[side][4] = at[side][4];
          q[side][5] = at[side][5];
        }
      }
      if (stale) // reload the top while the children are in flight
        reload();
#pragma unroll
      for (int side = 0; side < 2; side++)
        if (leaf[side] && ok[side])
          isect_f64<MODE>(q[side], idx[side], o, d, rtmin, rtmax, best);
      // The box tests of both sides, on a leaf's side without effect: no
      // divergence, and a box test is cheaper than the branches around it.
      bool hit2[2];
      double tn2[2];
      uint2 g2[2];
#pragma unroll
      for (int side = 0; side < 2; side++) {
        const double2 b0 = q[side][0], b1 = q[side][1], b2 = q[side][2], b3 = q[side][3];
        const double lo[3] = { b0.x, b0.y, b1.x };
        const double hi[3] = { b1.y, b2.x, b2.y };
        g2[side] = make_uint2(pack(uint64_t(__double_as_longlong(b3.x))),
                              pack(uint64_t(__double_as_longlong(b3.y))));
        double tn[3], tf[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
          double nb = pos_dir[k] ? lo[k] : hi[k];
          double fb = pos_dir[k] ? hi[k] : lo[k];
          double pn = nb * rcp[k];
          tn[k] = pn + ipos[k];
          double pf = fb * rcp[k];
          tf[k] = pf + ipos[k];
        }
        const double tmin = dm_max(dm_max(tn[0], tn[1]), tn[2]);
        const double tmax = dm_min(dm_min(tf[0], tf[1]), tf[2]);
        // tmax >= max(0, tmin), false for a NaN on either side
        hit2[side] = !leaf[side] && ok[side] && (tmax >= tmin) && (tmax >= 0.0);
        tn2[side] = tmin;
      }
      const bool left_first = hit2[0] && (!hit2[1] || tn2[0] < tn2[1]);
      const double next_t = left_first ? tn2[0] : tn2[1];
      ch[0] = left_first ? g2[0].x : g2[1].x;
      ch[1] = left_first ? g2[0].y : g2[1].y;
      // push-then-pop of the near child: its push needs room; its pop is then
      // pruned when a closer hit is already known
      bool have = hit2[0] || hit2[1];
      if (hit2[0] && hit2[1] && sp < uint32_t(kStackF64)) {
        push(make_uint2(left_first ? g2[1].x : g2[0].x, left_first ? g2[1].y : g2[0].y),
             left_first ? tn2[1] : tn2[0]);
      }
      have = have && sp < uint32_t(kStackF64) && !(best.t < next_t);
      // Pruned entries are dropped here, one after another: a trip round the
      // outer loop for each would wait for the other lanes' visits.
      while (!have && sp > 0) {
        if (stale)
          reload();
        sp--;
        stale = sp > 0;
        ch[0] = top_lr.x;
        ch[1] = top_lr.y;
        have = !(best.t < top_t);
      }
      // Every lane meets here before the next visit: without it the compiler
      // lets the lanes that already have a node loop on alone.
      __builtin_amdgcn_wave_barrier();
      if (!have)
        break;
    }
  }
  const bool hit = best.prim != ~uint64_t(0);
  prim_out[i] = best.prim;
  t_out[i] = best.t;
  if (uv_out)
    *reinterpret_cast<double2*>(uv_out + 2 * i) = make_double2(hit ? best.u : 0.0,
                                                               hit ? best.v : 0.0);
}

} // namespace lbvh_dev

namespace lbvh_eng {

using namespace lbvh_dev;

hipError_t
launch_trace_f64(int mode, const void* nodes, const double* tris, uint64_t n,
                 const double* rays, uint64_t nrays, uint64_t* prim, double* t, double* uv,
                 hipStream_t s)
{
  if (nrays == 0)
    return hipSuccess;
  const uint32_t g = uint32_t((nrays + kTraceF64Block - 1) / kTraceF64Block);
  const Node64* nd = static_cast<const Node64*>(nodes);
  if (mode == 0)
    hipLaunchKernelGGL((k_trace_f64<0>), dim3(g), dim3(kTraceF64Block), 0, s, nd, tris, n, rays,
                       nrays, prim, t, uv);
  else if (mode == 1)
    hipLaunchKernelGGL((k_trace_f64<1>), dim3(g), dim3(kTraceF64Block), 0, s, nd, tris, n, rays,
                       nrays, prim, t, uv);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

} // namespace lbvh_eng
