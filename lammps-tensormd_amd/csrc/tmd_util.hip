// Small device kernels: buffer clearing (a kernel, so it is safe inside
// captured graphs), and what follows the force kernel: fixed-order FP64
// reductions of energy/virial and kinetic energy with the second half of the
// velocity-Verlet step (src/fix_nve.cpp:102-130).
#include "tmd_desc_common.h"

#include <algorithm>

namespace tmd {

namespace {

__global__ void k_zero(uint4 *p, size_t n16, unsigned char *tail, size_t ntail)
{
  size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t) gridDim.x * blockDim.x;
  for (size_t q = i; q < n16; q += stride) p[q] = make_uint4(0, 0, 0, 0);
  if (i < ntail) tail[i] = 0;
}

// What the end of a step needs of memory, requested before the sums.
struct StepEnd {
  Ctl ctl;
  unsigned long long n;
};

__device__ inline StepEnd load_end(const StepTail &a)
{
  StepEnd e{};
  if (a.ctl) e.ctl = load_ctl(a.ctl);
  if (a.hist) e.n = a.counter[0];
  return e;
}

// tot[0..7] = energy, virial, sum m v^2 (held by the workgroup) -> results
__device__ inline void finish_step(const StepTail &a, StepEnd &end, const double *tot)
{
  const int t = threadIdx.x;
  if (t < 7) a.out[t] = tot[t];
  if (t != 0) return;
  if (a.ctl) {
    reset_ctl(a.ctl, end.ctl, a.trig2);
    if (a.ctl_host)
      for (int q = 0; q < 4; q++) a.ctl_host[q] = end.ctl.w[q];
  }
  if (a.hist) {
    const unsigned long long n = end.n;
    if (n < (unsigned long long) a.hist_cap) {
      a.hist[2 * n] = tot[0];
      a.hist[2 * n + 1] = 0.5 * 1.0364269e-4 * tot[7];  // mvv2e, metal units
    }
    a.counter[0] = n + 1;
  }
}

// Sums over the atoms, and the second half of a velocity-Verlet step
// (src/fix_nve.cpp:102-130) in the same pass.  Each workgroup writes its
// partial sums, added in a fixed order by k_step_final; the only workgroup
// of a small system finishes by itself.
__global__ __launch_bounds__(1024) void k_step_sums(StepTail a)
{
  __shared__ double sh[16][8];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nw = blockDim.x >> 6;
  StepEnd end{};
  if (gridDim.x == 1 && t == 0) end = load_end(a);
  double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 2
  for (int i = blockIdx.x * blockDim.x + t; i < a.n; i += gridDim.x * blockDim.x) {
    s[0] += a.eatom[i];
#pragma unroll
    for (int q = 0; q < 6; q++) s[1 + q] += a.watom[6 * (size_t) i + q];
    if (a.v) {
      const int e = (int) a.pos[i].w;
      const double c = a.dtfm[e];
      double v2 = 0.0;
#pragma unroll
      for (int q = 0; q < 3; q++) {
        const size_t p = 3 * (size_t) i + q;
        const double v = a.v[p] + c * a.f[p];
        a.v[p] = v;
        v2 += v * v;
      }
      s[7] += a.mass[e] * v2;
    }
  }
  // pairs of quantities share the exchanges between halves and rows
  const double x0 = row_sum_d(swap16_add(swap32_add(s[0], s[1]), swap32_add(s[2], s[3])));
  const double x1 = row_sum_d(swap16_add(swap32_add(s[4], s[5]), swap32_add(s[6], s[7])));
  if ((lane & 15) == 0) {
    const int q = ((lane >> 4) & 1) * 2 + (lane >> 5);  // rows hold quantities 0, 2, 1, 3
    sh[wave][q] = x0;
    sh[wave][4 + q] = x1;
  }
  __syncthreads();
  double r = 0.0;
  if (t < 8)
    for (int w = 0; w < nw; w++) r += sh[w][t];
  if (gridDim.x > 1) {
    if (t < 8) a.out[8 + 8 * (size_t) blockIdx.x + t] = r;
    return;
  }
  __syncthreads();
  if (t < 8) sh[0][t] = r;
  __syncthreads();
  finish_step(a, end, sh[0]);
}

// one wave per quantity; fixed shuffle tree (deterministic)
__global__ __launch_bounds__(512) void k_step_final(StepTail a, int nparts)
{
  __shared__ double tot[8];
  const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
  StepEnd end{};
  if (threadIdx.x == 0) end = load_end(a);
  double s = 0.0;
  for (int p = lane; p < nparts; p += 64) s += a.out[8 + 8 * (size_t) p + q];
  s = wave_sum_d(s);
  if (lane == 0) tot[q] = s;
  __syncthreads();
  finish_step(a, end, tot);
}

__global__ void k_set_positions(int first, int n, const double *x, double4 *pos, unsigned long long *ctl)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) ctl[1] = 1ull;  // rebuild the list
  if (i >= n) return;
  double4 p = pos[first + i];
  p.x = x[3 * (size_t) i];
  p.y = x[3 * (size_t) i + 1];
  p.z = x[3 * (size_t) i + 2];
  pos[first + i] = p;
}

__global__ void k_copy_small(const double *src, double *dst, int n)
{
  if ((int) threadIdx.x < n) dst[threadIdx.x] = src[threadIdx.x];
}

// One thread per value, so that a wave writes 512 contiguous bytes.
__global__ void k_pack_state(int first, int n, StateOut s)
{
  const size_t n3 = 3 * (size_t) n, total = (s.pos ? n3 : 0) + (s.v ? n3 : 0) + (s.f ? n3 : 0) + (s.eatom ? n : 0);
  const size_t f3 = 3 * (size_t) first, stride = (size_t) gridDim.x * blockDim.x;
  for (size_t t = (size_t) blockIdx.x * blockDim.x + threadIdx.x; t < total; t += stride) {
    size_t q = t;
    double val = 0.0;
    bool done = false;
    if (s.pos) {
      if (q < n3) {
        val = reinterpret_cast<const double *>(s.pos + first + q / 3)[q % 3];
        done = true;
      } else {
        q -= n3;
      }
    }
    if (!done && s.v) {
      if (q < n3) {
        val = s.v[f3 + q];
        done = true;
      } else {
        q -= n3;
      }
    }
    if (!done && s.f) {
      if (q < n3) {
        val = s.f[f3 + q];
        done = true;
      } else {
        q -= n3;
      }
    }
    if (!done) val = s.eatom[first + q];
    s.out[t] = val;
  }
}

__global__ void k_snapshot(int n, bool save, double4 *pos, double *v, double *f, double4 *sp, double *sv, double *sf,
                           unsigned long long *counter)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) counter[0] = 0ull;
  if (i >= n) return;
  if (save)
    sp[i] = pos[i];
  else
    pos[i] = sp[i];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    const size_t k = (size_t) q * n + i;  // any order: both sides are [n][3]
    if (save) {
      sv[k] = v[k];
      sf[k] = f[k];
    } else {
      v[k] = sv[k];
      f[k] = sf[k];
    }
  }
}

__global__ void k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16)
{
  size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t) gridDim.x * blockDim.x;
  for (size_t q = i; q < n16; q += stride) dst[q] = src[q];
}

}  // namespace

hipError_t launch_copy(const void *src, void *dst, size_t bytes, hipStream_t s)
{
  size_t n16 = bytes / 16;
  k_copy<<<8192, 256, 0, s>>>((const uint4 *) src, (uint4 *) dst, n16);
  return hipGetLastError();
}

hipError_t launch_set_positions(int first, int n, const double *x, double4 *pos, unsigned long long *ctl,
                                hipStream_t s)
{
  if (n <= 0) return hipSuccess;
  k_set_positions<<<(n + 255) / 256, 256, 0, s>>>(first, n, x, pos, ctl);
  return hipGetLastError();
}

hipError_t launch_pack_state(int first, int n, const StateOut &o, hipStream_t s)
{
  const size_t total = (size_t) n * ((o.pos ? 3 : 0) + (o.v ? 3 : 0) + (o.f ? 3 : 0) + (o.eatom ? 1 : 0));
  if (total == 0) return hipSuccess;
  k_pack_state<<<(int) std::min<size_t>(2048, (total + 255) / 256), 256, 0, s>>>(first, n, o);
  return hipGetLastError();
}

hipError_t launch_copy_small(const double *src, double *dst, int n, hipStream_t s)
{
  k_copy_small<<<1, 64, 0, s>>>(src, dst, n);
  return hipGetLastError();
}

hipError_t launch_snapshot(int n, bool save, double4 *pos, double *v, double *f, void *snap,
                           unsigned long long *counter, hipStream_t s)
{
  double4 *sp = static_cast<double4 *>(snap);
  double *sv = reinterpret_cast<double *>(sp + n), *sf = sv + 3 * (size_t) n;
  k_snapshot<<<(n + 255) / 256, 256, 0, s>>>(n, save, pos, v, f, sp, sv, sf, counter);
  return hipGetLastError();
}

hipError_t launch_zero(void *p, size_t bytes, hipStream_t s)
{
  if (bytes == 0) return hipSuccess;
  size_t n16 = bytes / 16, tail = bytes - n16 * 16;
  int blocks = (int) std::min<size_t>(4096, (n16 + 255) / 256 + 1);
  k_zero<<<blocks, 256, 0, s>>>((uint4 *) p, n16, (unsigned char *) p + n16 * 16, tail);
  return hipGetLastError();
}

hipError_t launch_step_tail(const StepTail &t, hipStream_t s)
{
  // one workgroup up to 2,048 atoms: two atoms per thread cost less than a
  // second launch
  if (t.n <= 2048) {
    k_step_sums<<<1, 1024, 0, s>>>(t);
  } else {
    const int parts = std::min(kSumParts, (t.n + 255) / 256);
    k_step_sums<<<parts, 256, 0, s>>>(t);
    k_step_final<<<1, 512, 0, s>>>(t, parts);
  }
  return hipGetLastError();
}

// Sum of the kept-neighbor counts over the real rows (the first word of
// each row of the descriptor's kept-list cache), added to *acc: one atomic
// per wave.
__global__ void k_sum_kept(const uint32_t *kl, size_t words, const int *row2atom, int nrows,
                           unsigned long long *acc)
{
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long v = 0;
  if (r < nrows && row2atom[r] >= 0) v = kl[(size_t) r * words];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  if ((threadIdx.x & 63) == 0 && v) atomicAdd(acc, v);
}

hipError_t launch_sum_kept(const uint32_t *kl, size_t words, const int *row2atom, int nrows,
                           unsigned long long *acc, hipStream_t s)
{
  if (nrows <= 0) return hipSuccess;
  k_sum_kept<<<(nrows + 255) / 256, 256, 0, s>>>(kl, words, row2atom, nrows, acc);
  return hipGetLastError();
}

}  // namespace tmd
