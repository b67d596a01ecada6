// Device neighbor build for periodic cells (any triclinic cell).
//
// Replaces LAMMPS NPairFullBin::build (src/npair_full_bin.cpp:68-126) with
// binning (src/nbin_standard.cpp:82-160) and the displacement trigger of
// Neighbor::decide/check_distance (src/neighbor.cpp:2293-2360, triggersq at
// :344).  The full list keeps every (j, image) with |d|^2 <= (rc+skin)^2,
// i != j or a non-zero image (npair_full_bin.cpp:99).  Bins are cells of the
// fractional lattice; a stencil of (2*reach+1)^3 bins reaches every
// candidate, including several periodic images when the cell is small.
//
// The rebuild decision is taken on the device: every kernel here reads the
// control word and exits when no rebuild is due, so a step never waits for
// the host.
//
// One launch serves a batch of independent structures: each atom carries
// its cell (atom_struct), each cell owns a contiguous range of global bins,
// and the stencil of an atom only visits its own cell's bins, so atoms of
// different structures never see each other.
#include "tmd_device.h"

#include <algorithm>

namespace tmd {

namespace {

__device__ inline void displacement(const double4 &xi, const double4 &xj, int s0, int s1, int s2,
                                    const CellInfo &c, double d[3])
{
#pragma clang fp contract(off)
  // Same expression, same order as the oracle: (xj - xi) + ((s0 h0 + s1 h1) + s2 h2)
  double sh0 = ((double) s0 * c.h[0] + (double) s1 * c.h[3]) + (double) s2 * c.h[6];
  double sh1 = ((double) s0 * c.h[1] + (double) s1 * c.h[4]) + (double) s2 * c.h[7];
  double sh2 = ((double) s0 * c.h[2] + (double) s1 * c.h[5]) + (double) s2 * c.h[8];
  d[0] = (xj.x - xi.x) + sh0;
  d[1] = (xj.y - xi.y) + sh1;
  d[2] = (xj.z - xi.z) + sh2;
}

__device__ inline double dist2(const double d[3])
{
#pragma clang fp contract(off)
  return d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
}

__device__ inline const CellInfo &cell_of(const NbrBuild &nb, int i)
{
  return nb.cells[nb.atom_struct ? nb.atom_struct[i] : 0];
}

__device__ inline int live_atoms(const NbrBuild &nb) { return nb.dyn ? nb.dyn->natoms : nb.n; }
__device__ inline int live_bins(const NbrBuild &nb, int nbins) { return nb.dyn ? nb.dyn->nbins : nbins; }

__device__ inline bool rebuild_due(const unsigned long long *ctl, double trig2)
{
  double m = __longlong_as_double((long long) ctl[0]);
  return ctl[1] != 0ull || m > trig2;
}

// Inclusive sum over the lanes (DPP: shifts within rows of 16, then the row
// totals 15 -> 16.., 31 -> 32.. broadcast to the rows behind).
__device__ inline int wave_scan(int v)
{
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Clears the bin counts for a build that may follow in this step: part `id`
// of `stride` threads.  Runs in the kernel before the build's first one.
__device__ inline void clear_bins(const NbrBuild &nb, int id, int stride)
{
  const int nbins = live_bins(nb, nb.nbins);
  for (int b = id; b < nbins; b += stride) nb.bin_count[b] = 0;
  if (id == 0) *nb.bin_total = 0;
}

// ctl[0] = the largest d2 of the workgroups whose largest exceeds the trigger
// (as ordered bits of a positive double): no one else's matters, and one
// atomic per workgroup on one word cost 5 us at 128,000 atoms.
__device__ inline void report_move(double d2, double trig2, unsigned long long *ctl)
{
  for (int o = 32; o > 0; o >>= 1) d2 = fmax(d2, __shfl_xor(d2, o));
  __shared__ double wmax[16];
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = d2;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = 0.0;
    for (int w = 0; w < (int) (blockDim.x >> 6); w++) m = fmax(m, wmax[w]);
    if (m > trig2) atomicMax(&ctl[0], (unsigned long long) __double_as_longlong(m));
  }
}

__device__ inline double moved2(const NbrBuild &nb, int i, const double4 &p)
{
  const double dx = p.x - nb.x_build[4 * (size_t) i], dy = p.y - nb.x_build[4 * (size_t) i + 1],
               dz = p.z - nb.x_build[4 * (size_t) i + 2];
  return dx * dx + dy * dy + dz * dz;
}

// max |x - x_build|^2 over atoms, and the bin counts cleared
__global__ void k_nb_check(NbrBuild nb, const double4 *pos)
{
  const int n = live_atoms(nb);
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  clear_bins(nb, i, gridDim.x * blockDim.x);
  report_move(i < n ? moved2(nb, i, pos[i]) : 0.0, nb.trig2, nb.ctl);
}

// First half of a velocity-Verlet step of one atom (src/fix_nve.cpp:64-98),
// its force cleared for the force kernel; returns its displacement^2 since the build.
__device__ inline double vv_atom(const NbrBuild &nb, int i, double4 *pos, double *v, double *f, const double *dtfm,
                                 double dt)
{
  double4 p = pos[i];
  const double c = dtfm[(int) p.w];
  const size_t q = 3 * (size_t) i;
  const double vx = v[q] + c * f[q], vy = v[q + 1] + c * f[q + 1], vz = v[q + 2] + c * f[q + 2];
  v[q] = vx;
  v[q + 1] = vy;
  v[q + 2] = vz;
  f[q] = f[q + 1] = f[q + 2] = 0.0;
  p.x += dt * vx;
  p.y += dt * vy;
  p.z += dt * vz;
  pos[i] = p;
  return moved2(nb, i, p);
}

// That half step with the displacement check of the new positions.
__global__ void k_vv_first(NbrBuild nb, int n, double4 *pos, double *v, double *f, const double *dtfm, double dt)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  clear_bins(nb, i, gridDim.x * blockDim.x);
  report_move(i < n ? vv_atom(nb, i, pos, v, f, dtfm, dt) : 0.0, nb.trig2, nb.ctl);
}

// wrap atom i into its cell, remember its build position; returns its bin
__device__ inline int bin_atom(const NbrBuild &nb, double4 *pos, int i)
{
  const CellInfo &c = cell_of(nb, i);
  double4 p = pos[i];
  double f[3];
  f[0] = p.x * c.inv[0] + p.y * c.inv[3] + p.z * c.inv[6];
  f[1] = p.x * c.inv[1] + p.y * c.inv[4] + p.z * c.inv[7];
  f[2] = p.x * c.inv[2] + p.y * c.inv[5] + p.z * c.inv[8];
  double s[3] = {floor(f[0]), floor(f[1]), floor(f[2])};
  if (s[0] != 0.0 || s[1] != 0.0 || s[2] != 0.0) {
    p.x -= (s[0] * c.h[0] + s[1] * c.h[3]) + s[2] * c.h[6];
    p.y -= (s[0] * c.h[1] + s[1] * c.h[4]) + s[2] * c.h[7];
    p.z -= (s[0] * c.h[2] + s[1] * c.h[5]) + s[2] * c.h[8];
    pos[i] = p;
    for (int a = 0; a < 3; a++) f[a] -= s[a];
  }
  nb.x_build[4 * (size_t) i + 0] = p.x;
  nb.x_build[4 * (size_t) i + 1] = p.y;
  nb.x_build[4 * (size_t) i + 2] = p.z;
  int b[3];
  for (int a = 0; a < 3; a++) {
    int q = (int) floor(f[a] * c.nb[a]);
    b[a] = min(max(q, 0), c.nb[a] - 1);
    nb.atom_bc[3 * (size_t) i + a] = b[a];
  }
  return c.bin_base + (b[0] * c.nb[1] + b[1]) * c.nb[2] + b[2];
}

// An atom and its position at its place in the bin-sorted order: w holds
// the index (exact in FP64).
__device__ inline double4 sorted_entry(const double4 &p, int i) { return make_double4(p.x, p.y, p.z, (double) i); }

// ---- bins of a large system: one kernel per phase ----
// Each atom's bin, and an arrival rank within it (any order).
__global__ void k_nb_bin(NbrBuild nb, double4 *pos)
{
  if (!rebuild_due(nb.ctl, nb.trig2)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= live_atoms(nb)) return;
  const int flat = bin_atom(nb, pos, i);
  nb.atom_bin[i] = flat;
  nb.atom_rank[i] = atomicAdd(&nb.bin_count[flat], 1);
}

// Room for every bin's atoms: consecutive within 64 bins, the groups of 64
// in any order (one counter update per group; the list kernel reads bins
// through their starts, so their order does not reach the list).
__global__ void k_nb_alloc(NbrBuild nb, int nbins)
{
  if (!rebuild_due(nb.ctl, nb.trig2)) return;
  const int b = blockIdx.x * blockDim.x + threadIdx.x, lane = threadIdx.x & 63;
  const bool in = b < live_bins(nb, nbins);
  const int cnt = in ? nb.bin_count[b] : 0;
  const int incl = wave_scan(cnt);
  int base = 0;
  if (lane == 63) base = atomicAdd(nb.bin_total, incl);
  base = __shfl(base, 63);
  if (in) nb.bin_start[b] = base + incl - cnt;
}

__global__ void k_nb_fill(NbrBuild nb)
{
  if (!rebuild_due(nb.ctl, nb.trig2)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= live_atoms(nb)) return;
  nb.bin_atoms[nb.bin_start[nb.atom_bin[i]] + nb.atom_rank[i]] = i;
}

// Ascending atom index inside each bin (a deterministic order): an atom's
// place is the number of smaller indices among its bin's atoms.
__global__ void k_nb_sort(NbrBuild nb, const double4 *pos)
{
  if (!rebuild_due(nb.ctl, nb.trig2)) return;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= live_atoms(nb)) return;
  const int b = nb.atom_bin[i], lo = nb.bin_start[b], cnt = nb.bin_count[b];
  int r = 0;
  for (int q = 0; q < cnt; q++) r += nb.bin_atoms[lo + q] < i ? 1 : 0;
  nb.sorted[lo + r] = sorted_entry(pos[i], i);
}

// ---- bins of a small system: the same phases in one workgroup ----
constexpr int kSmall = 4096;  // atoms and bins at most
// Atoms up to which the workgroup also takes the first half of an MD step:
// two atoms per thread cost less than a launch of their own.
constexpr int kSmallStep = 2048;

bool small_build(const NbrBuild &nb) { return nb.n <= kSmall && nb.nbins <= kSmall; }
bool small_step(const NbrBuild &nb) { return small_build(nb) && nb.n <= kSmallStep && !nb.dyn; }

template <bool VV>
__global__ __launch_bounds__(1024) void k_nb_small(NbrBuild nb, double4 *pos, int nbins, double *v, double *f,
                                                   const double *dtfm, double dt)
{
  __shared__ int count[kSmall], start[kSmall], atoms[kSmall], wsum[16];
  if constexpr (VV) {
    const bool flagged = rebuild_due(nb.ctl, nb.trig2);
    double d2 = 0.0;
#pragma unroll
    for (int u = 0; u < kSmallStep / 1024; u++) {
      const int i = u * 1024 + (int) threadIdx.x;
      if (i < nb.n) d2 = fmax(d2, vv_atom(nb, i, pos, v, f, dtfm, dt));
    }
    const bool moved = __syncthreads_or(d2 > nb.trig2);
    if (moved) report_move(d2, nb.trig2, nb.ctl);  // the list kernel reads it
    if (!flagged && !moved) return;
  } else if (!rebuild_due(nb.ctl, nb.trig2)) {
    return;
  }
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int n = min(live_atoms(nb), kSmall);
  nbins = min(live_bins(nb, nbins), kSmall);
  for (int b = t; b < kSmall; b += 1024) count[b] = 0;
  __syncthreads();
  int bin[kSmall / 1024], rank[kSmall / 1024];
#pragma unroll
  for (int u = 0; u < kSmall / 1024; u++) {
    const int i = u * 1024 + t;
    bin[u] = rank[u] = 0;
    if (i < n) {
      bin[u] = min(bin_atom(nb, pos, i), kSmall - 1);
      rank[u] = atomicAdd(&count[bin[u]], 1);
    }
  }
  __syncthreads();
  // exclusive scan, 4 consecutive bins per thread
  int c[4], sum = 0;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    c[u] = count[4 * t + u];
    sum += c[u];
  }
  const int incl = wave_scan(sum);
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wave; w++) run += wsum[w];
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int b = 4 * t + u;
    start[b] = run;
    if (b < nbins) {
      nb.bin_start[b] = run;
      nb.bin_count[b] = c[u];
    }
    run += c[u];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kSmall / 1024; u++) {
    const int i = u * 1024 + t;
    if (i < n) atoms[start[bin[u]] + rank[u]] = i;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kSmall / 1024; u++) {
    const int i = u * 1024 + t;
    if (i >= n) continue;
    const int lo = start[bin[u]], cnt = count[bin[u]];
    int r = 0;
    for (int q = 0; q < cnt; q++) r += atoms[lo + q] < i ? 1 : 0;
    nb.sorted[lo + r] = sorted_entry(pos[i], i);
  }
}

// floor(a / b) for |a|, b < 2^20, ib = 1 / b: a + 1/2 is at least 1 / (2 b)
// away from a multiple of b, relative to which the rounding of the product is
// small.
__device__ inline int small_div(int a, float ib) { return (int) floorf(((float) a + 0.5f) * ib); }

// One wavefront per atom.  Its stencil bins (in the order o0, o1, o2) are
// read one per lane; the lanes write their bins' places in the sorted order
// to LDS behind one another (a prefix sum of the counts), and the wave then
// takes 64 of these candidates at a time: one contiguous 32-byte load per
// lane, and a ballot places the kept ones.  The list order is the serial
// walk's: stencil order, then ascending atom index within a bin.
// Workgroups of the list kernel at most: they stride over the atoms, so that
// the steps without a rebuild do not launch one wave per atom to return.
constexpr int kListBlocks = 4096;
constexpr int kCand = 768;  // candidates held in LDS per wave; longer stencils take several rounds

__global__ __launch_bounds__(256) void k_nb_list(NbrBuild nb, const double4 *pos, uint32_t *nbr, int *nn)
{
  if (!rebuild_due(nb.ctl, nb.trig2)) return;
  __shared__ uint32_t s_cand[4][kCand];
  const int lane = threadIdx.x & 63;
  uint32_t *cand = s_cand[threadIdx.x >> 6];
  const int n = live_atoms(nb);
  for (int i = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)); i < n; i += 4 * gridDim.x) {
    const CellInfo &c = cell_of(nb, i);
    const double4 xi = pos[i];
    const int bc0 = nb.atom_bc[3 * (size_t) i], bc1 = nb.atom_bc[3 * (size_t) i + 1],
              bc2 = nb.atom_bc[3 * (size_t) i + 2];
    const int n0 = c.nb[0], n1 = c.nb[1], n2 = c.nb[2];
    const int w2 = 2 * c.reach[2] + 1, w12 = (2 * c.reach[1] + 1) * w2;
    const int nst = (2 * c.reach[0] + 1) * w12;
    const float iw2 = 1.0f / (float) w2, iw12 = 1.0f / (float) w12;
    const float in0 = 1.0f / (float) n0, in1 = 1.0f / (float) n1, in2 = 1.0f / (float) n2;
    uint32_t *out = nbr + (size_t) i * nb.cap;
    int base = 0;    // entries written so far (wave-uniform)
    int ncand = 0;   // candidates held in LDS (wave-uniform)
    auto flush = [&]() {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      // four loads per lane in flight: the wave waits for memory, not for arithmetic
      for (int t0 = 0; t0 < ncand; t0 += 256) {
        uint32_t e[4];
        double4 xj[4];
#pragma unroll
        for (int u = 0; u < 4; u++) e[u] = cand[min(t0 + 64 * u + lane, ncand - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++) xj[u] = nb.sorted[e[u] & kNbrJMask];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (t0 + 64 * u >= ncand) break;
          const uint32_t code = e[u] >> kNbrJBits;
          double d[3] = {xj[u].x - xi.x, xj[u].y - xi.y, xj[u].z - xi.z};
          // most waves of a large cell hold no image: nothing to decode or add
          if (__builtin_amdgcn_ballot_w64(code != kShiftCenter) != 0ull) {
            const int s0 = (int) (code / 49u) - 3, s1 = (int) ((code / 7u) % 7u) - 3, s2 = (int) (code % 7u) - 3;
            displacement(xi, xj[u], s0, s1, s2, c, d);
          }
          const int j = (int) xj[u].w;
          const bool keep = t0 + 64 * u + lane < ncand && dist2(d) <= nb.cut2 && !(j == i && code == kShiftCenter);
          const unsigned long long m = __ballot(keep);
          const int k = base + (int) __builtin_amdgcn_mbcnt_hi((unsigned) (m >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((unsigned) m, 0u));
          if (keep && k < nb.cap) out[k] = (uint32_t) j | (code << kNbrJBits);
          base += __popcll(m);
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      ncand = 0;
    };
    for (int r0 = 0; r0 < nst; r0 += 64) {
      const int sidx = r0 + lane;
      int lo = 0, cnt = 0;
      uint32_t code = 0;
      if (sidx < nst) {
        const int i0 = small_div(sidx, iw12), rem = sidx - i0 * w12, i1 = small_div(rem, iw2);
        const int q0 = bc0 + i0 - c.reach[0], q1 = bc1 + i1 - c.reach[1], q2 = bc2 + rem - i1 * w2 - c.reach[2];
        const int s0 = small_div(q0, in0), s1 = small_div(q1, in1), s2 = small_div(q2, in2);
        const int t0 = q0 - s0 * n0, t1 = q1 - s1 * n1, t2 = q2 - s2 * n2;
        const int b = c.bin_base + (t0 * n1 + t1) * n2 + t2;
        lo = nb.bin_start[b];
        cnt = nb.bin_count[b];
        code = (uint32_t) ((s0 + 3) * 49 + (s1 + 3) * 7 + (s2 + 3)) << kNbrJBits;
      }
      // these bins' candidates in order, as many at a time as fit
      const int incl = wave_scan(cnt);
      const int excl = incl - cnt, total = __builtin_amdgcn_readlane(incl, 63);
      if (ncand + total > kCand) flush();
      for (int w0 = 0; w0 < total; w0 += kCand) {  // one pass unless the round alone overfills LDS
        const int wend = min(total, w0 + kCand);
        const int q0 = max(0, w0 - excl), q1 = min(cnt, wend - excl);
        for (int q = q0; q < q1; q++) cand[ncand + excl + q - w0] = (uint32_t) (lo + q) | code;
        ncand += wend - w0;
        if (wend < total) flush();
      }
    }
    flush();
    if (lane == 0) {
      nn[i] = min(base, nb.cap);
      if (base > nb.cap) atomicMax(&nb.ctl[2], (unsigned long long) base);
    }
  }
}

}  // namespace

hipError_t nbr_check(const NbrBuild &nb, const double4 *pos, hipStream_t stream)
{
  if (nb.n <= 0) return hipSuccess;
  k_nb_check<<<(nb.n + 1023) / 1024, 1024, 0, stream>>>(nb, pos);
  return hipGetLastError();
}

hipError_t launch_vv_first(const NbrBuild &nb, int n, double4 *pos, double *v, double *f, const double *dtfm,
                           double dt, hipStream_t stream)
{
  if (n == nb.n && small_step(nb))
    k_nb_small<true><<<1, 1024, 0, stream>>>(nb, pos, nb.nbins, v, f, dtfm, dt);
  else
    k_vv_first<<<(n + 255) / 256, 256, 0, stream>>>(nb, n, pos, v, f, dtfm, dt);
  return hipGetLastError();
}

hipError_t nbr_rebuild(const NbrBuild &nb, double4 *pos, uint32_t *nbr, int *nn, hipStream_t stream, bool after_vv)
{
  if (nb.n <= 0) return hipSuccess;
  const int blocks = (nb.n + 255) / 256;
  if (after_vv && small_step(nb)) {
    // binned by launch_vv_first
  } else if (small_build(nb)) {
    k_nb_small<false><<<1, 1024, 0, stream>>>(nb, pos, nb.nbins, nullptr, nullptr, nullptr, 0.0);
  } else {
    k_nb_bin<<<blocks, 256, 0, stream>>>(nb, pos);
    k_nb_alloc<<<(nb.nbins + 255) / 256, 256, 0, stream>>>(nb, nb.nbins);
    k_nb_fill<<<blocks, 256, 0, stream>>>(nb);
    k_nb_sort<<<blocks, 256, 0, stream>>>(nb, pos);
  }
  k_nb_list<<<std::min((nb.n + 3) / 4, kListBlocks), 256, 0, stream>>>(nb, pos, nbr, nn);
  return hipGetLastError();
}

}  // namespace tmd
