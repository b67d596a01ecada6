// Staging kernels of the batched single-point path.  One kernel copies a
// packed batch (pinned host memory, read directly by the GPU) into the
// slot's fixed device arrays and one writes the results back, so a batch is
// a single graph launch with no memcpy nodes and no host round trips.
//
// Every count and index read from the staging area is clamped to the slot
// capacities before any kernel uses it; a clamp sets an error flag that the
// host reads back with the results.
#include "tmd_desc_common.h"

#include <algorithm>

namespace tmd {

namespace {

// The batch's extents, clamped to the capacities; pad is set if one was not
// within them.
__device__ inline BatchDims clamp_header(const unsigned char *stage, const BatchCaps &caps)
{
  BatchDims d = *reinterpret_cast<const BatchDims *>(stage);
  int err = 0;
  auto clampi = [&err](int v, int hi) {
    if (v < 0 || v > hi) {
      err = 1;
      return v < 0 ? 0 : hi;
    }
    return v;
  };
  d.natoms = clampi(d.natoms, caps.atoms);
  d.nstruct = clampi(d.nstruct, caps.structs);
  d.nbins = clampi(d.nbins, caps.bins);
  d.rl.nrows = clampi(d.rl.nrows, caps.rows);
  // element row groups: non-decreasing, empty beyond the model's elements
  int prev = 0;
  for (int e = 0; e <= kMaxElts; e++) {
    int v = clampi(d.rl.row_off[e], d.rl.nrows);
    if (v < prev || (e >= caps.nelt && v != d.rl.nrows && e > 0)) {
      err = 1;
      v = e >= caps.nelt ? d.rl.nrows : prev;
    }
    d.rl.row_off[e] = v;
    prev = v;
  }
  if (d.rl.row_off[0] != 0) err = 1;
  d.rl.row_off[0] = 0;
  d.pad = err;
  return d;
}

// Staging -> device arrays.  Host memory is far (1.5-2 us a trip), so every
// workgroup reads the header itself instead of waiting for a kernel that does,
// and a thread's first entry of every array is requested before any is used.
// One structure of 54 atoms: 4.3 (header kernel) + 10.4 us -> 7.9 us.
__global__ __launch_bounds__(256) void k_batch_unpack(const unsigned char *stage, BatchCaps caps, BatchArrays a)
{
  __shared__ BatchDims head;
  if (threadIdx.x == 0) head = clamp_header(stage, caps);
  __syncthreads();
  const BatchDims &d = head;
  const int ns = d.nstruct, n = d.natoms, nr = d.rl.nrows;
  size_t off[7];
  batch_stage_offsets(ns, n, nr, off);
  const unsigned char *body = stage + sizeof(BatchDims);
  const int *soff = reinterpret_cast<const int *>(body);
  const CellInfo *cells = reinterpret_cast<const CellInfo *>(stage + off[1]);
  const int *as = reinterpret_cast<const int *>(stage + off[2]);
  const int *r2a = reinterpret_cast<const int *>(stage + off[3]);
  const double4 *pos = reinterpret_cast<const double4 *>(stage + off[4]);
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const int stride = gridDim.x * blockDim.x;
  int bad = 0;
  if (tid == 0) {
    *a.dyn = d;
    a.ctl[1] = 1ull;  // every batch builds its neighbor list
  }
  // clamped, unconditional first loads: a masked one would be waited for at
  // the end of its branch
  const int soff0 = soff[min(tid, ns)], as0 = as[min(tid, max(n - 1, 0))], r0 = r2a[min(tid, max(nr - 1, 0))];
  const double4 p0 = pos[min(tid, max(n - 1, 0))];
  auto put_offset = [&](int q, int v) {
    if (v < 0 || v > n) bad = 1;
    a.struct_off[q] = min(max(v, 0), n);
  };
  auto put_struct = [&](int q, int s) {
    if (s < 0 || s >= ns) {
      bad = 1;
      s = 0;
    }
    a.atom_struct[q] = s;
  };
  auto put_row = [&](int q, int i) {
    if (i >= n) {
      bad = 1;
      i = -1;
    }
    a.row2atom[q] = i < 0 ? -1 : i;
  };
  auto put_pos = [&](int q, double4 p) {
    if (!(p.w >= 0.0 && p.w < (double) caps.nelt)) {
      bad = 1;
      p.w = 0.0;
    }
    a.pos[q] = p;
  };
  for (int q = tid; q < ns; q += stride) {
    CellInfo c = cells[q];
    long nb = 1;
    for (int k = 0; k < 3; k++) {
      if (c.nb[k] < 1 || c.nb[k] > 1024 || c.reach[k] < 0 || c.reach[k] > 64) {
        bad = 1;
        c.nb[k] = 1;
        c.reach[k] = 0;
      }
      nb *= c.nb[k];
    }
    if (c.bin_base < 0 || c.bin_base + nb > d.nbins) {
      bad = 1;
      c.nb[0] = c.nb[1] = c.nb[2] = 1;
      c.reach[0] = c.reach[1] = c.reach[2] = 0;
      c.bin_base = 0;
    }
    a.cells[q] = c;
  }
  if (tid <= ns) put_offset(tid, soff0);
  if (tid < n) put_struct(tid, as0);
  if (tid < nr) put_row(tid, r0);
  if (tid < n) put_pos(tid, p0);
  for (int q = tid + stride; q <= ns; q += stride) put_offset(q, soff[q]);
  for (int q = tid + stride; q < n; q += stride) put_struct(q, as[q]);
  for (int q = tid + stride; q < nr; q += stride) put_row(q, r2a[q]);
  for (int q = tid + stride; q < n; q += stride) put_pos(q, pos[q]);
  // cleared for this batch's list build and force sums
  for (int q = tid; q < 3 * n; q += stride) a.f[q] = 0.0;
  for (int q = tid; q < d.nbins; q += stride) a.bin_count[q] = 0;
  if (tid == 0) *a.bin_total = 0;
  if (bad) atomicOr(&a.ctl[5], 1ull);
}

// sums of eatom[i], watom[i][0..5] over atoms [lo, hi) by one 256-thread
// workgroup, in a fixed order; thread 0..6 of the result hold the 7 sums
__device__ inline void block_sum7(const double *eatom, const double *watom, int lo, int hi,
                                  int stride_lo, int stride, double (*sh)[256], double *res)
{
  int t = threadIdx.x;
  double v[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int i = lo + stride_lo + t; i < hi; i += stride) {
    v[0] += eatom[i];
    for (int q = 0; q < 6; q++) v[1 + q] += watom[(size_t) i * 6 + q];
  }
  for (int q = 0; q < 7; q++) sh[q][t] = v[q];
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (t < o)
      for (int q = 0; q < 7; q++) sh[q][t] += sh[q][t + o];
    __syncthreads();
  }
  if (t < 7) res[t] = sh[t][0];
}

// Results -> host memory: forces and energies by all workgroups, then each
// structure's sums by one.  (As two kernels, sums and copy: 4.5 + 4.0 us for
// one structure of 54 atoms; now 4.1 us.)
__global__ __launch_bounds__(256) void k_batch_finish(double *out, BatchArrays a)
{
  __shared__ double sh[7][256];
  const int ns = a.dyn->nstruct, n = a.dyn->natoms;
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  const int stride = gridDim.x * blockDim.x;
  if (tid == 0) {
    Ctl c = load_ctl(a.ctl);
    out[0] = (double) c.w[2];
    out[1] = (double) n;
    out[2] = (double) ns;
    out[3] = a.dyn->pad != 0 || a.ctl[5] != 0ull ? 1.0 : 0.0;
    for (int q = 4; q < 8; q++) out[q] = 0.0;
    reset_ctl(a.ctl, c, 0.0);
    a.ctl[2] = 0ull;
    a.ctl[5] = 0ull;
  }
  double *so = out + 8;
  double *fo = so + 7 * (size_t) ns;
  double *eo = fo + 3 * (size_t) n;
  for (int q = tid; q < 3 * n; q += stride) fo[q] = a.f[q];
  for (int q = tid; q < n; q += stride) eo[q] = a.eatom[q];
  for (int st = blockIdx.x; st < ns; st += gridDim.x) {
    __syncthreads();
    block_sum7(a.eatom, a.watom, a.struct_off[st], a.struct_off[st + 1], 0, 256, sh, so + 7 * (size_t) st);
  }
}

int grid_for(long work)
{
  long b = (work + 255) / 256;
  return (int) (b < 1 ? 1 : (b > 1024 ? 1024 : b));
}

}  // namespace

hipError_t launch_batch_unpack(const void *stage, const BatchCaps &caps, const BatchArrays &a,
                               hipStream_t stream)
{
  const unsigned char *st = static_cast<const unsigned char *>(stage);
  long work = caps.atoms > caps.rows ? caps.atoms : caps.rows;
  k_batch_unpack<<<grid_for(work), 256, 0, stream>>>(st, caps, a);
  return hipGetLastError();
}

hipError_t launch_batch_finish(void *out, const BatchCaps &caps, const BatchArrays &a,
                               hipStream_t stream)
{
  const int blocks = std::max(grid_for(3L * caps.atoms), std::min(caps.structs, 1024));
  k_batch_finish<<<blocks, 256, 0, stream>>>(static_cast<double *>(out), a);
  return hipGetLastError();
}

}  // namespace tmd
