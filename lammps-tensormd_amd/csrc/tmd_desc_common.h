// Device helpers shared by the descriptor and force kernels
// (tmd_desc.hip: max_moment 0-3; tmd_desc_hm.hip: max_moment 4-5):
// periodic displacements, the Kerley interpolation, wave reductions, the
// slot-sorted compaction of an atom's list and per-neighbor geometry.
#pragma once
#include "tmd_device.h"

namespace tmd {

namespace {

// Lattice rows of the cell an atom belongs to (uniform per workgroup).
struct Box {
  double h[9];
};

__device__ inline Box load_box(const Geom &geo, int i)
{
  const CellInfo &c = geo.cells[geo.atom_struct ? geo.atom_struct[i] : 0];
  Box b;
#pragma unroll
  for (int q = 0; q < 9; q++) b.h[q] = c.h[q];
  return b;
}

__device__ inline void displacement(const double4 &xi, const double4 &xj, uint32_t code,
                                    const Box &c, double d[3])
{
#pragma clang fp contract(off)
  d[0] = xj.x - xi.x;
  d[1] = xj.y - xi.y;
  d[2] = xj.z - xi.z;
  // no image shift in the whole wave (list mode, and most atoms of a large
  // cell): nothing to decode or add
  if (__builtin_amdgcn_ballot_w64(code != kShiftCenter) == 0ull) return;
  int s0 = (int) (code / 49u) - 3, s1 = (int) ((code / 7u) % 7u) - 3, s2 = (int) (code % 7u) - 3;
  double sh0 = ((double) s0 * c.h[0] + (double) s1 * c.h[3]) + (double) s2 * c.h[6];
  double sh1 = ((double) s0 * c.h[1] + (double) s1 * c.h[4]) + (double) s2 * c.h[7];
  double sh2 = ((double) s0 * c.h[2] + (double) s1 * c.h[5]) + (double) s2 * c.h[8];
  d[0] += sh0;
  d[1] += sh1;
  d[2] += sh2;
}

__device__ inline double dist2(const double d[3])
{
#pragma clang fp contract(off)
  return d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
}

// Kerley rational interpolation of one filter (gpu/cuda/ration.cu:59-68) in
// units of the grid step: table entry t = (y, s dx, c1 dx^2, c2 dx^2),
// q = r / dx - n, p = 1 - q, qp = q - p:
//   w = |c2 p| / (|c2 p| + |c1 q|)  (0 when both vanish)
//   c = c2 + w (c1 - c2),  h = y + q (s - p c),
//   dx dh/dr = s + (q - p) c + w (1 - w) (c1 - c2)
// (the last term is the reference's dx (c - c2)(1 - w)).  Evaluated through
// 1 - w = |c1 q| / den: the smallest normal number added to |c1 q| makes the
// denominator positive and 1 - w = 1 when both vanish, and is lost in
// rounding otherwise.
__device__ inline float kerley_w1(float4 t, float q, float p)
{
  const float b = fmaf(fabsf(t.z), fabsf(q), 1.17549435e-38f);
  return b * __builtin_amdgcn_rcpf(fmaf(fabsf(t.w), fabsf(p), b));  // 1-ulp reciprocal
}

__device__ inline float kerley_h(float4 t, float q, float p)
{
  const float c = fmaf(kerley_w1(t, q, p), t.w - t.z, t.z);
  return fmaf(q, fmaf(-p, c, t.y), t.x);
}

__device__ inline void kerley(float4 t, float q, float p, float qp, float &h, float &dxdh)
{
  const float w = kerley_w1(t, q, p);
  const float dc = t.w - t.z;
  const float c = fmaf(w, dc, t.z);
  h = fmaf(q, fmaf(-p, c, t.y), t.x);
  dxdh = fmaf(dc, fmaf(w, w, -w), fmaf(qp, c, t.y));
}

// Cross-lane moves within a row of 16 lanes (DPP: no LDS traffic).
// quad_perm [1,0,3,2] and [2,3,0,1] swap lanes 2i <-> 2i+1 and i <-> i^2;
// row_ror:4 and row_ror:8 rotate a row of 16 lanes.
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppRor4 = 0x124, kDppRor8 = 0x128;

template <int CTRL>
__device__ inline double dpp_d(double v)
{
  long long b = __double_as_longlong(v);
  int lo = __builtin_amdgcn_mov_dpp((int) (b & 0xffffffffll), CTRL, 0xF, 0xF, false);
  int hi = __builtin_amdgcn_mov_dpp((int) (b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long) hi << 32) | (unsigned int) lo);
}

// Sum over the 64 lanes, the result in every lane (fixed order: the same
// lanes combine in the same order on every call).
__device__ inline double wave_sum_d(double v)
{
  v += dpp_d<kDppXor1>(v);
  v += dpp_d<kDppXor2>(v);
  v += dpp_d<kDppRor4>(v);
  v += dpp_d<kDppRor8>(v);
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

// a's lanes 0-31 + 32-63 in lanes 0-31, b's in lanes 32-63
__device__ inline float swap32_add(float a, float b)
{
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// rows of 16 lanes: row 0 of the result = a's rows 0 + 1, row 1 = b's rows
// 0 + 1, row 2 = a's rows 2 + 3, row 3 = b's rows 2 + 3
__device__ inline float swap16_add(float a, float b)
{
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ inline double make_d(unsigned lo, unsigned hi)
{
  return __longlong_as_double((long long) (((unsigned long long) hi << 32) | lo));
}

__device__ inline double swap32_add(double a, double b)
{
  const unsigned long long ua = (unsigned long long) __double_as_longlong(a), ub = (unsigned long long) __double_as_longlong(b);
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned) ua, (unsigned) ub, false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned) (ua >> 32), (unsigned) (ub >> 32), false, false);
  return make_d(l[0], h[0]) + make_d(l[1], h[1]);
}

__device__ inline double swap16_add(double a, double b)
{
  const unsigned long long ua = (unsigned long long) __double_as_longlong(a), ub = (unsigned long long) __double_as_longlong(b);
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned) ua, (unsigned) ub, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned) (ua >> 32), (unsigned) (ub >> 32), false, false);
  return make_d(l[0], h[0]) + make_d(l[1], h[1]);
}

// Orders LDS accesses of the workgroup's only wave: its LDS instructions run
// in order, so the compiler must keep the order and nothing has to be waited
// for.
__device__ inline void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ inline double row_sum_d(double v)
{
  v += dpp_d<kDppXor1>(v);
  v += dpp_d<kDppXor2>(v);
  v += dpp_d<kDppRor4>(v);
  v += dpp_d<kDppRor8>(v);
  return v;
}

__device__ inline unsigned lane_rank(unsigned long long m)
{
  return __builtin_amdgcn_mbcnt_hi((unsigned) (m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned) m, 0u));
}

// Phase 1: compact the kept entries (slot-sorted).  start[b] .. start[b+1].
__device__ inline int kept_slot(const ModelGeo &g, const Box &cell, const double4 &xi, int ei,
                                uint32_t e, const double4 &xj, double d[3])
{
  displacement(xi, xj, e >> kNbrJBits, cell, d);
  double r2 = dist2(d);
  return (r2 < g.rc2 && r2 > 1e-10) ? (int) ((g.slots[ei] >> (4 * (int) xj.w)) & 15u)
                                    : -1;  // kernel.cu:1163
}

__device__ inline int kept_slot(const ModelGeo &g, const Box &cell, const double4 &xi, int ei,
                                uint32_t e, const double4 &xj)
{
  double d[3];
  return kept_slot(g, cell, xi, ei, e, xj, d);
}

// Lists of at most 64 NCH entries: every entry's slot stays in registers.
// All loads are unconditional, with indices clamped into the row (and to
// atom 0 past its end), and issued before any is used: exec-masked loads
// make the compiler wait for each one at its branch join.
template <int NCH>
__device__ inline int compact_short(const ModelGeo &g, const Box &cell, const double4 &xi, int ei,
                                    const uint32_t *list, int nraw, const double4 *pos,
                                    uint32_t *kept, int *start)
{
  const int lane = threadIdx.x & 63;
  const int last = max(nraw - 1, 0);
  uint32_t ent[NCH];
  double4 xj[NCH];
  int slot[NCH];
#pragma unroll
  for (int ch = 0; ch < NCH; ch++) {
    const int idx = ch * 64 + lane;
    const uint32_t e = list[min(idx, last)];
    ent[ch] = idx < nraw ? e : 0u;
  }
#pragma unroll
  for (int ch = 0; ch < NCH; ch++) xj[ch] = pos[ent[ch] & kNbrJMask];
#pragma unroll
  for (int ch = 0; ch < NCH; ch++) {
    const int sl = kept_slot(g, cell, xi, ei, ent[ch], xj[ch]);
    slot[ch] = ch * 64 + lane < nraw ? sl : -1;
  }
  int s = 0;
  for (int b = 0; b < g.nelt; b++) {
    start[b] = s;
#pragma unroll
    for (int ch = 0; ch < NCH; ch++) s += __popcll(__ballot(slot[ch] == b));
  }
  start[g.nelt] = s;
  for (int b = 0; b < g.nelt; b++) {
    int run = start[b];
#pragma unroll
    for (int ch = 0; ch < NCH; ch++) {
      unsigned long long m = __ballot(slot[ch] == b);
      if (slot[ch] == b) kept[run + (int) lane_rank(m)] = ent[ch];
      run += __popcll(m);
    }
  }
  return s;
}

__device__ inline int compact(const ModelGeo &g, const Box &cell, const double4 &xi, int ei,
                              const uint32_t *list, int nraw, const double4 *pos, uint32_t *kept,
                              int *start)
{
  const int lane = threadIdx.x & 63;
  if (nraw <= 128) return compact_short<2>(g, cell, xi, ei, list, nraw, pos, kept, start);
  if (nraw <= 192) return compact_short<3>(g, cell, xi, ei, list, nraw, pos, kept, start);
  if (nraw <= 256) return compact_short<4>(g, cell, xi, ei, list, nraw, pos, kept, start);
  // long lists: two sweeps
  int cnt[kMaxElts];
  for (int b = 0; b < kMaxElts; b++) cnt[b] = 0;
  for (int base = 0; base < nraw; base += 64) {
    int idx = base + lane, slot = -1;
    if (idx < nraw) {
      uint32_t e = list[idx];
      slot = kept_slot(g, cell, xi, ei, e, pos[e & kNbrJMask]);
    }
    for (int b = 0; b < g.nelt; b++) cnt[b] += __popcll(__ballot(slot == b));
  }
  int s = 0;
  for (int b = 0; b < g.nelt; b++) {
    start[b] = s;
    s += cnt[b];
  }
  start[g.nelt] = s;
  int run[kMaxElts];
  for (int b = 0; b < kMaxElts; b++) run[b] = start[b];
  for (int base = 0; base < nraw; base += 64) {
    int idx = base + lane, slot = -1;
    uint32_t e = 0;
    if (idx < nraw) {
      e = list[idx];
      slot = kept_slot(g, cell, xi, ei, e, pos[e & kNbrJMask]);
    }
    for (int b = 0; b < g.nelt; b++) {
      unsigned long long m = __ballot(slot == b);
      if (slot == b) kept[run[b] + (int) lane_rank(m)] = e;
      run[b] += __popcll(m);
    }
  }
  return s;
}

// 1/sqrt(r2) in FP64: hardware estimate plus one Newton step (relative
// error ~1e-15, far below the FP32 arithmetic that uses it)
__device__ inline double rsqrt_fp64(double r2)
{
  double y = __builtin_amdgcn_rsq(r2);
  return y * (1.5 - 0.5 * r2 * y * y);
}

// Geometry of one kept neighbor: FP64 displacement, unit vector and r, and
// the radial-table cell n with the offsets q = r / dx - n, 1 - q
// (ration.cu:29-32).
struct NbrGeo {
  double d[3];
  double r;
  float ux, uy, uz;
  float q, pq;
  int n, j;
};

// from the displacement o.d
__device__ inline void nbr_geometry(const ModelGeo &g, NbrGeo &o)
{
  double r2 = o.d[0] * o.d[0] + o.d[1] * o.d[1] + o.d[2] * o.d[2];
  double rinv = rsqrt_fp64(r2);
  o.r = r2 * rinv;
  o.ux = (float) (o.d[0] * rinv);
  o.uy = (float) (o.d[1] * rinv);
  o.uz = (float) (o.d[2] * rinv);
  o.n = min(g.tab_n - 2, (int) (o.r * g.xdx));
  const double qd = o.r * g.rdx - (double) o.n;
  o.q = (float) qd;
  o.pq = (float) (1.0 - qd);
}

__device__ inline void nbr_geometry(const ModelGeo &g, const Box &cell, const double4 &xi,
                                    const double4 *pos, uint32_t e, NbrGeo &o)
{
  o.j = (int) (e & kNbrJMask);
  displacement(xi, pos[o.j], e >> kNbrJBits, cell, o.d);
  nbr_geometry(g, o);
}

// the end cells of the table are zero (ration.hpp:29)
__device__ inline bool table_cell_live(const ModelGeo &g, int n) { return n > 0 && n < g.tab_n - 2; }

// The control word of the neighbor list after an evaluation: a build counted
// if one was due, flags cleared for the next step.
struct Ctl {
  unsigned long long w[4];
};

__device__ inline Ctl load_ctl(const unsigned long long *ctl)
{
  Ctl c;
  for (int q = 0; q < 4; q++) c.w[q] = ctl[q];
  return c;
}

__device__ inline void reset_ctl(unsigned long long *ctl, Ctl &c, double trig2)
{
  if (c.w[1] != 0ull || __longlong_as_double((long long) c.w[0]) > trig2) ctl[3] = ++c.w[3];
  c.w[0] = c.w[1] = 0ull;
  ctl[0] = 0ull;
  ctl[1] = 0ull;
}

}  // namespace

}  // namespace tmd
