// Closest-hit traversal on gfx950.
//
// Reproduces traverser::operator() (lbvh.h:1874-1942) exactly: the root is
// pushed with tmin = +inf; a popped entry is skipped when the closest hit so
// far is nearer than its tmin; leaf children are intersected at once, left
// then right; internal children get the octant slab test (make_accel_ray,
// lbvh.h:991-1010; detail::intersect, lbvh.h:1071-1091; hit iff
// tmax >= max(0, tmin), lbvh.h:1023-1026) and are pushed far first, near
// last; the stack holds 128 entries and drops pushes when full
// (traversal_stack<float,128>, lbvh.h:1746-1789).
//
// It walks the reference's node array itself.  A node is visited with its
// two children already known (they came with its own record, loaded when its
// box was tested), so one round of independent loads serves a visit: the
// 32-byte record of an internal child (its box and its children) and the
// 48-byte triangle of a leaf child are fetched together.  A pushed node
// carries its children on the stack.
#include "device_common.hpp"
#include "engine.hpp"

namespace lbvh_dev {

using lbvh_eng::TraceJob;

// Two waves per workgroup: measured faster than four (the clustered 1M
// primary launch 0.68 -> 0.65 ms) and the same as one.
constexpr int kTraceBlock = 128;
// The occupancy knob's "no limit" (the registers then allow what they allow).
constexpr int kTraceMaxWavesPerSimd = 8;
constexpr int kStack = 128;
// Stack entries kept in LDS (12 bytes each; a power of two, a ring): 12 KB
// per workgroup.  2,073,600 primary / 148,743 bounce rays on the clustered 1M
// scene with rings of 4, 8 and 16 entries: 525 / 447, 518 / 420 and 675 / 417
// us (16 leave three waves per SIMD).
constexpr int kStackLds = 8;
// s_waitcnt operand: no vector memory operation outstanding (vmcnt 0, other
// counters at their maximum).
constexpr int kWaitVmem0 = 0x0F70;

struct Ray
{
  float o[3];
  float d[3];
  float tmin, tmax;
};

// lbvh::math::dot (lbvh.h:621-630): accumulation starts from 0.
__device__ __forceinline__ float
dot3(const float* a, const float* b)
{
  float out = 0.0f;
  float px = a[0] * b[0];
  out = out + px;
  float py = a[1] * b[1];
  out = out + py;
  float pz = a[2] * b[2];
  out = out + pz;
  return out;
}

// lbvh::math::cross (lbvh.h:609-616)
__device__ __forceinline__ void
cross3(const float* a, const float* b, float* o)
{
  float ay_bz = a[1] * b[2], az_by = a[2] * b[1];
  float az_bx = a[2] * b[0], ax_bz = a[0] * b[2];
  float ax_by = a[0] * b[1], ay_bx = a[1] * b[0];
  o[0] = ay_bz - az_by;
  o[1] = az_bx - ax_bz;
  o[2] = ax_by - ay_bx;
}

struct Tri
{
  float p0[3], e0[3], e1[3], nrm[3];
};

// The closest hit so far.
struct Hit
{
  uint32_t prim = 0xffffffffu;
  float t = INFINITY, u = 0.0f, v = 0.0f;
};

// Whether a hit at distance t of primitive id replaces the closest so far.
template<int MODE>
__device__ __forceinline__ bool
better(float t, uint32_t id, const Hit& h)
{
  if (MODE == 0)
    return t < h.t;
  return (t < h.t) || (t == h.t && id < h.prim && t != INFINITY);
}

// triangle_intersector (lbvh.h:2055-2075): two-sided, not watertight.
template<int MODE>
__device__ __forceinline__ void
isect_reference(const Tri& tr, uint32_t id, const Ray& r, Hit& h)
{
  float c[3] = { tr.p0[0] - r.o[0], tr.p0[1] - r.o[1], tr.p0[2] - r.o[2] };
  float rr[3];
  cross3(r.d, c, rr);
  float inv_det = 1.0f / dot3(tr.nrm, r.d);
  float u = dot3(rr, tr.e1) * inv_det;
  float v = dot3(rr, tr.e0) * inv_det;
  float w = (1.0f - u) - v;
  if ((u >= 0.0f) && (v >= 0.0f) && (w >= 0.0f)) {
    float t = dot3(tr.nrm, c) * inv_det;
    if ((t >= r.tmin) && (t <= r.tmax) && better<MODE>(t, id, h)) {
      h.prim = id;
      h.t = t;
      h.u = u;
      h.v = v;
    }
  }
}

// Watertight test (Woop, Benthin, Wald, JCGT 2(1) 2013) on A = p0,
// B = p0 - e0, C = p0 + e1; u, v are the weights of B and C.
template<int MODE>
__device__ __forceinline__ void
isect_watertight(const Tri& tr, uint32_t id, const Ray& r, Hit& h)
{
  float ax = fabsf(r.d[0]), ay = fabsf(r.d[1]), az = fabsf(r.d[2]);
  int kz = (ax > ay) ? ((ax > az) ? 0 : 2) : ((ay > az) ? 1 : 2);
  int kx = (kz == 2) ? 0 : kz + 1;
  int ky = (kx == 2) ? 0 : kx + 1;
  float dkz = r.d[0], dkx = r.d[0], dky = r.d[0];
  // component selects without dynamic register indexing
  auto comp = [](const float* v, int k) { return k == 0 ? v[0] : (k == 1 ? v[1] : v[2]); };
  dkz = comp(r.d, kz);
  if (dkz < 0.0f) {
    int tmp = kx;
    kx = ky;
    ky = tmp;
  }
  dkx = comp(r.d, kx);
  dky = comp(r.d, ky);
  float Sx = dkx / dkz;
  float Sy = dky / dkz;
  float Sz = 1.0f / dkz;
  float va[3], vb[3], vc[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    float b = tr.p0[k] - tr.e0[k];
    float c = tr.p0[k] + tr.e1[k];
    va[k] = tr.p0[k] - r.o[k];
    vb[k] = b - r.o[k];
    vc[k] = c - r.o[k];
  }
  float az_ = comp(va, kz), bz_ = comp(vb, kz), cz_ = comp(vc, kz);
  float sxa = Sx * az_, sya = Sy * az_;
  float sxb = Sx * bz_, syb = Sy * bz_;
  float sxc = Sx * cz_, syc = Sy * cz_;
  float Ax = comp(va, kx) - sxa, Ay = comp(va, ky) - sya;
  float Bx = comp(vb, kx) - sxb, By = comp(vb, ky) - syb;
  float Cx = comp(vc, kx) - sxc, Cy = comp(vc, ky) - syc;
  float cb = Cx * By, cyb = Cy * Bx;
  float U = cb - cyb;
  float acy = Ax * Cy, ayc = Ay * Cx;
  float V = acy - ayc;
  float bay = Bx * Ay, bya = By * Ax;
  float W = bay - bya;
  if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f))
    return;
  float det = U + V;
  det = det + W;
  if (det == 0.0f)
    return;
  float Az = Sz * az_, Bz = Sz * bz_, Cz = Sz * cz_;
  float ua = U * Az, vb2 = V * Bz, wc = W * Cz;
  float T = ua + vb2;
  T = T + wc;
  float rcp = 1.0f / det;
  float t = T * rcp;
  if (!(t >= r.tmin && t <= r.tmax && better<MODE>(t, id, h)))
    return;
  h.prim = id;
  h.t = t;
  h.u = V * rcp;
  h.v = W * rcp;
}

// Ray layouts: kLayoutSingle, one tree; kLayoutBatch, a scene batch (ray i
// belongs to the scene s with ray_off[s] <= i < ray_off[s + 1], whose nodes
// start at prim_off[s] - s and whose triangles start at prim_off[s]; ids are
// scene-local); kLayoutJobs, independent trees with their own ray and output
// buffers (job k covers global rays [jobs[k].ray_begin, jobs[k + 1].ray_begin)).
constexpr int kLayoutSingle = 0;
constexpr int kLayoutBatch = 1;
constexpr int kLayoutJobs = 2;

// The last job with ray_begin <= i.
__device__ __forceinline__ uint32_t
job_of(const TraceJob* __restrict__ jobs, uint32_t njobs, uint64_t i)
{
  uint32_t lo = 0, hi = njobs;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (jobs[mid].ray_begin <= i)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// order (single layout only, may be null): ray k of the launch is ray
// order[k] of the input, and its hit is written there; a permutation that
// puts rays which visit the same nodes into the same wave.
//
// Bound by instruction issue (a vector instruction takes a SIMD four cycles
// for its 64 rays) and by the dependent fetch of each visit.  So a visit has
// no branch around loads, box tests or addresses (157 instead of 250 vector
// instructions), and a ray drops its pruned entries in a loop of its own
// instead of one per visit of its wave.  Clustered 1M scene, 2,073,600
// primary / 148,743 bounce rays: 621 / 546 us with branches per child, a trip
// per pruned entry and an LDS stack of the 6 entries nearest the root, 518 /
// 420 us so.
template<int MODE, int LAYOUT>
__global__ __launch_bounds__(kTraceBlock) void
k_trace(const Node* __restrict__ nodes, const float* __restrict__ tris, uint32_t nprims,
        const uint64_t* __restrict__ prim_off, const uint64_t* __restrict__ ray_off,
        uint32_t nseg, const TraceJob* __restrict__ jobs, const float* __restrict__ rays,
        const uint32_t* __restrict__ order, uint64_t nrays, uint32_t* __restrict__ prim_out,
        float* __restrict__ t_out, float* __restrict__ uv_out)
{
  // batches and jobs: the ray offsets of the scenes / jobs this workgroup's
  // rays fall in, staged once (s_rb) when they are at most kTraceBlock
  constexpr bool kStage = LAYOUT != kLayoutSingle;
  __shared__ uint64_t s_rb[kStage ? kTraceBlock + 1 : 1];
  __shared__ uint32_t s_first, s_span;
  const uint64_t i0 = uint64_t(blockIdx.x) * kTraceBlock;
  uint64_t i = i0 + threadIdx.x;
  uint32_t first = 0, span = 0;
  if constexpr (kStage) {
    if (threadIdx.x == 0) {
      const uint64_t last = (i0 + kTraceBlock <= nrays ? i0 + kTraceBlock : nrays) - 1;
      uint32_t a, b;
      if constexpr (LAYOUT == kLayoutBatch) {
        a = find_scene(ray_off, nseg, int64_t(i0), 1, false);
        b = find_scene(ray_off, nseg, int64_t(last), 1, false);
      } else {
        a = job_of(jobs, nseg, i0);
        b = job_of(jobs, nseg, last);
      }
      s_first = a;
      s_span = (b - a + 1 <= uint32_t(kTraceBlock)) ? b - a + 1 : 0u; // 0: not staged
    }
    __syncthreads();
    first = s_first;
    span = s_span;
    for (uint32_t t = threadIdx.x; t < span; t += kTraceBlock)
      s_rb[t] = (LAYOUT == kLayoutBatch) ? ray_off[first + t] : jobs[first + t].ray_begin;
    __syncthreads();
  }
  if (i >= nrays)
    return;
  uint32_t sel = 0; // the ray's scene or job
  if constexpr (kStage) {
    if (span) {
      uint32_t lo = 0, hi = span; // s_rb[lo] <= i, the last such entry
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (s_rb[mid] <= i)
          lo = mid;
        else
          hi = mid;
      }
      sel = first + lo;
    } else {
      sel = (LAYOUT == kLayoutBatch) ? find_scene(ray_off, nseg, int64_t(i), 1, false)
                                     : job_of(jobs, nseg, i);
    }
  }
  if constexpr (LAYOUT == kLayoutBatch) {
    const uint32_t sc = sel;
    const uint64_t P = prim_off[sc];
    nprims = uint32_t(prim_off[sc + 1] - P);
    nodes += P - sc;
    tris += 12 * P;
  } else if constexpr (LAYOUT == kLayoutJobs) {
    const TraceJob& jb = jobs[sel];
    nodes = static_cast<const Node*>(jb.nodes);
    tris = jb.tris;
    nprims = jb.nprims;
    rays = jb.rays;
    prim_out = jb.prim;
    t_out = jb.t;
    uv_out = jb.uv;
    i -= jb.ray_begin;
  } else {
    if (order)
      i = order[i];
  }
  const float4* rp = reinterpret_cast<const float4*>(rays + 8 * i);
  const float4 r0 = rp[0], r1 = rp[1];
  Ray r;
  r.o[0] = r0.x;
  r.o[1] = r0.y;
  r.o[2] = r0.z;
  r.d[0] = r0.w;
  r.d[1] = r1.x;
  r.d[2] = r1.y;
  r.tmin = r1.z;
  r.tmax = r1.w;

  // make_accel_ray
  float rcp[3], ipos[3];
  bool pos_dir[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    rcp[k] = 1.0f / r.d[k];
    float np = -r.o[k];
    ipos[k] = np * rcp[k];
    pos_dir[k] = r.d[k] > 0.0f;
  }

  // The traversal stack: capacity 128 with pushes dropped when full, as the
  // reference's.  An entry stands for a pushed node and holds what its own
  // node record gave when its box was tested: its two children and the box's
  // entry distance (the reference's tmin), so popping it needs no further
  // load.  The top entry is kept in registers: a pop hands it over at once
  // and leaves the register stale (stale: the top is still entry sp - 1); its
  // reload is issued after the children's fetches, so the latencies overlap,
  // and a push onto a stale top needs no reload at all.  Of the entries below
  // it, the kStackLds nearest the top are in an LDS ring (one column per
  // thread and field) and the first `low` in a private array: a ray at any
  // depth works in the ring, and goes to private memory only when it has
  // climbed or sunk by kStackLds entries.
  __shared__ uint32_t s_stk[3 * kStackLds * kTraceBlock];
  uint3 spill[kStack];
  uint32_t low = 0;
  auto ring = [&](uint32_t e) { return &s_stk[(e & (kStackLds - 1)) * kTraceBlock + threadIdx.x]; };
  auto ring_load = [&](uint32_t e) {
    const uint32_t* q = ring(e);
    return make_uint3(q[0], q[kStackLds * kTraceBlock], q[2 * kStackLds * kTraceBlock]);
  };
  uint3 top = make_uint3(0u, 0u, 0u);
  uint32_t sp = 0;
  bool stale = false;
  auto push = [&](uint3 v) {
    if (sp > 0 && !stale) {
      const uint32_t e = sp - 1;
      if (e - low == uint32_t(kStackLds)) {
        spill[low] = ring_load(low);
        low++;
      }
      uint32_t* q = ring(e);
      q[0] = top.x;
      q[kStackLds * kTraceBlock] = top.y;
      q[2 * kStackLds * kTraceBlock] = top.z;
    }
    stale = false;
    top = v;
    sp++;
  };
  auto reload = [&]() { // a stale top (sp > 0)
    const uint32_t e = sp - 1;
    if (e < low) {
      top = spill[e];
      low = e;
      // waited for here: left pending, it would make every later wait for a
      // child's data wait for more than that data
      __builtin_amdgcn_s_waitcnt(kWaitVmem0);
    } else {
      top = ring_load(e);
    }
    stale = false;
  };

  Hit best;

  // The reference pushes the root and pops it at once: its record gives the
  // first two children.  A node it would push and pop again straight away
  // (the near child, or a single hit child) is taken directly here, but only
  // when that push would have found room, so the visit order and the
  // drop-when-full rule are unchanged.
  if (nprims >= 2u) {
    const float4 root = reinterpret_cast<const float4*>(nodes)[1];
    uint32_t ch[2] = { __float_as_uint(root.z), __float_as_uint(root.w) };
    const char* const node_base = reinterpret_cast<const char*>(nodes);
    const char* const tri_base = reinterpret_cast<const char*>(tris);
    const uint32_t last_leaf = nprims - 1u, last_node = nprims - 2u;
    for (;;) {
      // Both children's data at once: a leaf's triangle, an internal node's
      // record (its box and children).  A child out of range (only possible
      // for a corrupt node array) is skipped; its loads go to the array's last
      // entry.  Offsets in 16-byte units: a node record is 2, a triangle 3.
      bool leaf[2], ok[2];
      uint32_t idx[2];
      float4 q0[2], q1[2], q2[2];
      const float4* at[2];
#pragma unroll
      for (int side = 0; side < 2; side++) {
        leaf[side] = int32_t(ch[side]) < 0;
        const uint32_t x = ch[side] & ~kLeafBit;
        const uint32_t lim = leaf[side] ? last_leaf : last_node;
        ok[side] = x <= lim;
        idx[side] = x < lim ? x : lim;
        const uint32_t units = idx[side] * 2u + (leaf[side] ? idx[side] : 0u);
        const char* base = leaf[side] ? tri_base : node_base;
        at[side] = reinterpret_cast<const float4*>(base + (uint64_t(units) << 4));
      }
#pragma unroll
      for (int side = 0; side < 2; side++) {
        q0[side] = at[side][0];
        q1[side] = at[side][1];
        if (leaf[side])
          q2[side] = at[side][2];
      }
      if (stale) // reload the top while the children are in flight
        reload();
#pragma unroll
      for (int side = 0; side < 2; side++) {
        if (!(leaf[side] && ok[side]))
          continue;
        const float4 a = q0[side], b = q1[side], c = q2[side];
        Tri tr;
        tr.p0[0] = a.x;
        tr.p0[1] = a.y;
        tr.p0[2] = a.z;
        tr.e0[0] = a.w;
        tr.e0[1] = b.x;
        tr.e0[2] = b.y;
        tr.e1[0] = b.z;
        tr.e1[1] = b.w;
        tr.e1[2] = c.x;
        tr.nrm[0] = c.y;
        tr.nrm[1] = c.z;
        tr.nrm[2] = c.w;
        if constexpr (MODE == 2)
          isect_watertight<MODE>(tr, idx[side], r, best);
        else
          isect_reference<MODE>(tr, idx[side], r, best);
      }
      // The box tests of both sides, on a leaf's side without effect: no
      // divergence, and a box test is cheaper than the branches around it.
      bool hit2[2];
      float tn2[2];
#pragma unroll
      for (int side = 0; side < 2; side++) {
        const float4 a = q0[side], b = q1[side];
        const float lo[3] = { a.x, a.y, a.z };
        const float hi[3] = { a.w, b.x, b.y };
        float tn[3], tf[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
          float nb = pos_dir[k] ? lo[k] : hi[k];
          float fb = pos_dir[k] ? hi[k] : lo[k];
          float pn = nb * rcp[k];
          tn[k] = pn + ipos[k];
          float pf = fb * rcp[k];
          tf[k] = pf + ipos[k];
        }
        const float tmin = m_max(m_max(tn[0], tn[1]), tn[2]);
        const float tmax = m_min(m_min(tf[0], tf[1]), tf[2]);
        // tmax >= max(0, tmin), false for a NaN on either side
        hit2[side] = !leaf[side] && ok[side] && (tmax >= tmin) && (tmax >= 0.0f);
        tn2[side] = tmin;
      }
      const bool left_first = hit2[0] && (!hit2[1] || tn2[0] < tn2[1]);
      const uint32_t gl0 = __float_as_uint(q1[0].z), gr0 = __float_as_uint(q1[0].w);
      const uint32_t gl1 = __float_as_uint(q1[1].z), gr1 = __float_as_uint(q1[1].w);
      const float next_t = left_first ? tn2[0] : tn2[1];
      ch[0] = left_first ? gl0 : gl1;
      ch[1] = left_first ? gr0 : gr1;
      // push-then-pop of the near child: its push needs room; its pop is then
      // pruned when a closer hit is already known
      bool have = hit2[0] || hit2[1];
      if (hit2[0] && hit2[1] && sp < uint32_t(kStack)) {
        push(make_uint3(left_first ? gl1 : gl0, left_first ? gr1 : gr0,
                        __float_as_uint(left_first ? tn2[1] : tn2[0])));
      }
      have = have && sp < uint32_t(kStack) && !(best.t < next_t);
      // Pruned entries are dropped here, one after another: a trip round the
      // outer loop for each would wait for the other lanes' visits.
      while (!have && sp > 0) {
        if (stale)
          reload();
        sp--;
        stale = sp > 0;
        ch[0] = top.x;
        ch[1] = top.y;
        have = !(best.t < __uint_as_float(top.z));
      }
      // Every lane meets here before the next visit: without it the compiler
      // lets the lanes that already have a node loop on alone (twice the
      // visits per wave, measured).
      __builtin_amdgcn_wave_barrier();
      if (!have)
        break;
    }
  }
  prim_out[i] = best.prim;
  t_out[i] = best.t;
  if (uv_out)
    *reinterpret_cast<float2*>(uv_out + 2 * i) = make_float2(best.u, best.v);
}

// ---- traversal order of a ray batch ---------------------------------------------
// Key of a ray: its direction octant (3 bits) above the 12-bit Morton code of
// the point o + d * reach, quantized to 16 cells per axis over the tree's
// centroid bounds grown by reach on every side, reach being the bounds'
// largest extent.  Rays with one key start in the same part of the scene and
// head the same way (for primary rays from one eye: neighbouring pixels), so
// a wave of them visits much the same nodes in the same order.  Sorted with
// two 8-bit radix passes; each workgroup encodes one chunk of the
// reduce-then-scan sort and writes that chunk's first-pass digit counts and
// its share of both passes' histograms (zero before).

constexpr int kRayKeyBlock = 256;

__device__ __forceinline__ uint32_t
spread4(uint32_t v)
{
  return (v & 1u) | ((v & 2u) << 2) | ((v & 4u) << 4) | ((v & 8u) << 6);
}

__global__ __launch_bounds__(kRayKeyBlock) void
k_ray_keys(const float* __restrict__ rays, uint64_t nrays, const float* __restrict__ bounds,
           uint32_t* __restrict__ keys, uint32_t* __restrict__ hist,
           uint32_t* __restrict__ counts, uint64_t chunk)
{
  __shared__ uint32_t s_hist[2 * 256];
  for (int j = threadIdx.x; j < 2 * 256; j += kRayKeyBlock)
    s_hist[j] = 0u;
  float lo[3], scale[3];
  float reach = 0.0f;
#pragma unroll
  for (int k = 0; k < 3; k++)
    reach = fmaxf(reach, bounds[3 + k] - bounds[k]);
  reach = fmaxf(reach, 1e-20f);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    lo[k] = bounds[k] - reach;
    scale[k] = 16.0f / (bounds[3 + k] + reach - lo[k]);
  }
  __syncthreads();
  const uint64_t b = uint64_t(blockIdx.x) * chunk;
  const uint64_t end = (b + chunk < nrays) ? b + chunk : nrays;
  for (uint64_t i = b + threadIdx.x; i < end; i += kRayKeyBlock) {
    const float4* rp = reinterpret_cast<const float4*>(rays + 8 * i);
    const float4 r0 = rp[0], r1 = rp[1];
    const float o[3] = { r0.x, r0.y, r0.z };
    const float d[3] = { r0.w, r1.x, r1.y };
    uint32_t q[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float p = o[k] + d[k] * reach;
      const float c = fminf(fmaxf((p - lo[k]) * scale[k], 0.0f), 15.0f); // NaN -> 0
      q[k] = uint32_t(c);
    }
    const uint32_t oct = (d[0] < 0.0f ? 4u : 0u) | (d[1] < 0.0f ? 2u : 0u) | (d[2] < 0.0f ? 1u : 0u);
    const uint32_t key = (oct << 12) | (spread4(q[0]) << 2) | (spread4(q[1]) << 1) | spread4(q[2]);
    keys[i] = key;
    atomicAdd(&s_hist[key & 0xffu], 1u);
    atomicAdd(&s_hist[256 + (key >> 8)], 1u);
  }
  __syncthreads();
  for (int j = threadIdx.x; j < 2 * 256; j += kRayKeyBlock) {
    const uint32_t v = s_hist[j];
    if (v)
      atomicAdd(&hist[j], v);
  }
  for (int dd = threadIdx.x; dd < 256; dd += kRayKeyBlock)
    counts[size_t(dd) * gridDim.x + blockIdx.x] = s_hist[dd];
}

} // namespace lbvh_dev

namespace lbvh_eng {

using namespace lbvh_dev;

// LDS a workgroup reserves beyond its own static `own` bytes so that at most
// `waves` waves share a SIMD: a workgroup puts its kTraceBlock / 64 waves on
// as many of the CU's 4 SIMDs, so that is waves * 4 / (kTraceBlock / 64)
// workgroups per CU, and one more must not fit.  0 = no limit beyond the
// registers'.
static size_t
occupancy_lds(int waves, size_t own)
{
  if (waves <= 0 || waves >= kTraceMaxWavesPerSimd)
    return 0;
  constexpr size_t kLdsPerCu = 160 * 1024;
  const size_t wgs = size_t(waves) * 4 / size_t(kTraceBlock / kWave);
  const size_t per_wg = (kLdsPerCu / wgs) & ~size_t(511);
  return per_wg > own ? per_wg - own : 0;
}

// Static LDS of a kernel, from its attributes (0 if they cannot be read; the
// failed query's error is cleared, so that it is not reported by the launch).
template<typename K>
static size_t
static_lds(K kernel)
{
  hipFuncAttributes a{};
  if (hipFuncGetAttributes(&a, reinterpret_cast<const void*>(kernel)) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return a.sharedSizeBytes;
}

template<int MODE>
static void
trace_mode(uint32_t g, int waves, hipStream_t s, const Node* nd, const float* tris,
           uint64_t n, const uint64_t* prim_off, const uint64_t* ray_off, uint32_t nseg,
           const TraceJob* jobs, const float* rays, const uint32_t* order, uint64_t nrays,
           uint32_t* prim, float* t, float* uv)
{
  static const size_t own_jobs = static_lds(k_trace<MODE, kLayoutJobs>);
  static const size_t own_batch = static_lds(k_trace<MODE, kLayoutBatch>);
  static const size_t own_single = static_lds(k_trace<MODE, kLayoutSingle>);
  if (jobs)
    hipLaunchKernelGGL((k_trace<MODE, kLayoutJobs>), dim3(g), dim3(kTraceBlock),
                       occupancy_lds(waves, own_jobs), s, nullptr, nullptr, 0u, nullptr, nullptr,
                       nseg, jobs, nullptr, nullptr, nrays, nullptr, nullptr, nullptr);
  else if (prim_off)
    hipLaunchKernelGGL((k_trace<MODE, kLayoutBatch>), dim3(g), dim3(kTraceBlock),
                       occupancy_lds(waves, own_batch), s, nd, tris, uint32_t(n), prim_off,
                       ray_off, nseg, nullptr, rays, nullptr, nrays, prim, t, uv);
  else
    hipLaunchKernelGGL((k_trace<MODE, kLayoutSingle>), dim3(g), dim3(kTraceBlock),
                       occupancy_lds(waves, own_single), s, nd, tris, uint32_t(n), nullptr,
                       nullptr, 1u, nullptr, rays, order, nrays, prim, t, uv);
}

static hipError_t
trace_dispatch(int mode, const void* nodes, const float* tris, uint64_t n, const uint64_t* prim_off,
               const uint64_t* ray_off, uint32_t nseg, const TraceJob* jobs, const float* rays,
               const uint32_t* order, uint64_t nrays, uint32_t* prim, float* t, float* uv,
               int waves, hipStream_t s)
{
  if (nrays == 0)
    return hipSuccess;
  const uint32_t g = uint32_t((nrays + kTraceBlock - 1) / kTraceBlock);
  const Node* nd = static_cast<const Node*>(nodes);
#define LBVH_TM(M)                                                                                \
  trace_mode<M>(g, waves, s, nd, tris, n, prim_off, ray_off, nseg, jobs, rays, order, nrays,       \
                prim, t, uv)
  switch (mode) {
    case 0:
      LBVH_TM(0);
      break;
    case 1:
      LBVH_TM(1);
      break;
    case 2:
      LBVH_TM(2);
      break;
    default:
      return hipErrorInvalidValue;
  }
#undef LBVH_TM
  return hipGetLastError();
}

hipError_t
launch_trace(int mode, const void* nodes, const float* tris, uint64_t n, const uint64_t* prim_off,
             const uint64_t* ray_off, uint32_t nseg, const float* rays, uint64_t nrays,
             uint32_t* prim, float* t, float* uv, hipStream_t s, const uint32_t* order,
             int waves_per_simd)
{
  if (prim_off && (!ray_off || nseg == 0))
    return hipErrorInvalidValue;
  if (prim_off && order)
    return hipErrorInvalidValue;
  return trace_dispatch(mode, nodes, tris, n, prim_off, ray_off, nseg, nullptr, rays, order, nrays,
                        prim, t, uv, waves_per_simd, s);
}

hipError_t
launch_trace_jobs(int mode, const TraceJob* jobs, uint32_t njobs, uint64_t nrays, hipStream_t s)
{
  if (!jobs || njobs == 0)
    return hipErrorInvalidValue;
  return trace_dispatch(mode, nullptr, nullptr, 0, nullptr, nullptr, njobs, jobs, nullptr, nullptr,
                        nrays, nullptr, nullptr, nullptr, 0, s);
}

hipError_t
launch_ray_keys(const float* rays, uint64_t nrays, const float* bounds, uint32_t* keys,
                uint32_t* hist, uint32_t* counts, uint32_t groups, uint64_t chunk, hipStream_t s)
{
  if (nrays == 0 || groups == 0 || chunk == 0 || uint64_t(groups) * chunk < nrays)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_ray_keys, dim3(groups), dim3(kRayKeyBlock), 0, s, rays, nrays, bounds,
                     keys, hist, counts, chunk);
  return hipGetLastError();
}

} // namespace lbvh_eng
