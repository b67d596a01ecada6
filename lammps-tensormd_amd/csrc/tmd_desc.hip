// Fused descriptor and force/virial kernels (gfx950, wave64), max_moment 0-3.
//
// One wavefront owns one atom.  The moments are carried in 16 real spherical
// harmonics Y_d(u) of degree 0..3 instead of the 20 monomials of the
// reference: on unit vectors the two span the same space, and with the
// normalisation of harmonics() the reference's tensor contractions are
//   G_0 = P_0                         G_1 = sum_{l=1} P_d^2
//   G_2 = P_0^2 / 3 + sum_{l=2} P_d^2     G_3 = 3/5 G_1 + sum_{l=3} P_d^2
// (cos^2 and cos^3 in Legendre polynomials and the addition theorem; a
// T-symmetric model drops the P_0^2 / 3 and 3/5 G_1 terms), where
// P[b][k][d] = sum over the neighbors c of slot b of H_k(r_c) Y_d(u_c).
//  1. Descriptor: sweep the atom's list (cutoff rc+skin) in chunks of 64,
//     keep 1e-10 < r^2 < rc^2 (gpu/cuda/kernel.cu:1163), find the element
//     slot b (tensormd.cpp:165-176) and compact the kept entries sorted by
//     slot (ballot prefix counts).  The force kernel reuses that list.
//  2. Staging: one lane per kept neighbor forms the FP64 geometry and writes
//     a row of LDS: its harmonics, and the radial-table cell and offsets.
//  3. Radial functions: 4 adjacent lanes per neighbor, 16 neighbors at a
//     time; for each of a lane's filters the 4 lanes read 64 contiguous
//     bytes of the table row (Kerley interpolation, gpu/cuda/ration.cu:13-71).
//     H goes through LDS into the operand layouts of the matrix cores.
//  4. P = Y^T H on v_mfma_f32_16x16x4_f32: 16 harmonics x 16 filters per
//     tile, 4 neighbors per instruction.
//     Force, slot by slot: S = dE/dP from P and dE/dG (kernel.cu:730-817),
//     then per tile of 16 neighbors U = S Y and V = S^T H on the matrix
//     cores, F = scale (sum_k U_k H'_k) u + scale V . dY/dd
//     (kernel.cu:559-646, :869-965); f_i += F, f_j -= F, virial -d (x) F
//     (kernel.cu:1714-1758), one lane per neighbor.
//
// MFMA operand layout (16x16x4): lane l holds A[l % 16][l / 16] and
// B[l / 16][l % 16]; accumulator element i of lane l is
// D[4 (l / 16) + i][l % 16].
//
// What bounds the kernels (128,000 atoms, 4 elements, 24 filters, 63
// neighbors): vector and matrix instructions, which do not overlap on a SIMD
// here, fill about 95 % of the force kernel's time (0.38 + 0.19 of 0.61 ms,
// single evaluations of the lattice; 0.42 ms with neither matrix instructions
// nor atomics) and 90 % of the descriptor's 0.30 ms.  With the monomials on
// the vector ALU they took 0.95 and 0.42 ms.  Along MD runs, which heat up, the
// force kernel's mean is 0.59 ms over 300 steps and 0.63 over 1,000 (69
// neighbors).
//
// Nothing per neighbor is stored in HBM: the reference materialises R, M,
// H, dH/dr, P, dE/dS, V, F1, F2 per padded slot (kernel.cu:1545-1582).
#include "tmd_desc_moments.h"

namespace tmd {

namespace {

template <int K, int NS, bool MP>
__global__ __launch_bounds__(64) void k_descriptor(ModelGeo g, Geom geo, const double4 *pos,
                                                   const uint32_t *nbr, const int *nn, int cap,
                                                   const int *row2atom, int rbase, int nrows,
                                                   const float4 *tab, float *G, uint32_t *kl)
{
  extern __shared__ __align__(16) unsigned char smem[];
  const int row = geo.order ? geo.order[rbase + (int) blockIdx.x] : rbase + (int) blockIdx.x;
  if (row >= nrows || (geo.dyn && row >= geo.dyn->rl.nrows)) return;
  float *Grow;
  const int i = descriptor_begin(g, geo, K, row, row2atom, G, Grow);
  if (i >= 0) descriptor_row<K, NS, MP>(g, geo, row, i, pos, nbr, nn, cap, tab, Grow, kl, smem);
}

// Waves per SIMD asked of the force kernel: what its LDS leaves room for.
// K = 32 spills 11 registers for it, and is still faster than at three waves
// or with one tile per slot in registers instead of two (Tiling::RT), neither
// of which spills (us, 1-2 elements, 62,500 atoms 250, 259 and 297; 65,536
// atoms 292, 304 and 288; eight elements, 65,536 atoms 532, 502 and 450).
template <int K>
constexpr int kForceWaves = K <= 32 ? 4 : (K == 64 ? 3 : 2);

template <int K>
__global__ __launch_bounds__(64, (kForceWaves<K>)) void k_force(ModelGeo g, Geom geo, const double4 *pos, int cap,
                                              const int *row2atom, int rbase, int nrows, const float4 *tab,
                                              const uint32_t *kl, const float *dEdG,
                                              const double *E, double scale, double *f,
                                              double *eatom, double *watom, double *vatom)
{
  using T = Tiling<K>;
  __shared__ __align__(16) float rows[T::WIN * kRow];
  __shared__ __align__(16) float buf[T::BUF];
  __shared__ double facc[9];
  const int row = geo.order ? geo.order[rbase + (int) blockIdx.x] : rbase + (int) blockIdx.x;
  if (row >= nrows || (geo.dyn && row >= geo.dyn->rl.nrows)) return;
  const int lane = threadIdx.x & 63;
  const int i = row2atom[row];
  if (i < 0) return;  // padding row
  float *hb = buf, *sb = T::kSRegs ? buf : buf + T::DBUF;
  const double4 xi = pos[i];
  const Box cell = load_box(geo, i);
  // the descriptor kernel's kept list of this row (slot-sorted, within rc):
  // the header in one register per lane, and the first two chunks' entries
  // read beside it (indices clamped into the row)
  const uint32_t *kr = kl + (size_t) row * kept_cache_words(cap);
  const uint32_t *kept = kr + kKeptHdr;
  const uint32_t hdr = kr[lane & 15];
  const uint32_t e0 = kept[min(lane, cap - 1)], e1 = kept[min(64 + lane, cap - 1)];
  const int nk = (int) __builtin_amdgcn_readlane((int) hdr, 0);
  auto start = [&](int b) { return (int) __builtin_amdgcn_readlane((int) hdr, 1 + b); };
  const float *grow = dEdG + (size_t) row * g.nelt * K * kNM;
  if (lane < 9) facc[lane] = 0.0;
  if (nk <= T::WIN) {
    // the whole list is staged at once; two lanes' worth of neighbors at most
    static_assert(T::WIN <= 128, "the list fits two chunks");
    double d0[3] = {0.0, 0.0, 0.0};
    if (lane < nk) stage_row(g, cell, xi, pos, e0, rows + lane * kRow, d0);
    if (64 + lane < nk) {
      double d1[3];
      stage_row(g, cell, xi, pos, e1, rows + (64 + lane) * kRow, d1);
    }
    wave_sync();
    auto next_slot = [&](int b) {
      while (b < g.nelt && start(b) >= start(b + 1)) b++;
      return b;
    };
    int b = next_slot(0);
    // the table rows of the next tile of filters are requested before the
    // present one goes through the matrix cores: the wave would otherwise
    // wait for them tile after tile
    TabTile<K> tt;
    auto request = [&](int bb) {
      if (T::RT > 0 && bb < g.nelt) load_tile<K>(tab, rows + start(bb) * kRow, min(16, start(bb + 1) - start(bb)), 0, tt);
    };
    request(b);
    while (b < g.nelt) {
      const int s0 = start(b), n = start(b + 1) - s0;
      const int bn = next_slot(b + 1);
      float *rt = rows + s0 * kRow;
      float4 gv[T::KT];
      load_dEdG<K>(grow + (size_t) b * K * kNM, gv);
      f32x4v acc[T::KT];
#pragma unroll
      for (int t = 0; t < T::KT; t++) acc[t] = f32x4v{0, 0, 0, 0};
      SOps<K> so;
      bool done = false;
      if constexpr (T::RT > 0) {
        // a slot of at most RT tiles: H and dH are interpolated once and stay
        // in registers between P and the chain rule
        if (n <= 16 * T::RT) {
          float h[T::RT][T::NFB], dh[T::RT][T::NFB];
#pragma unroll
          for (int q = 0; q < T::RT; q++) {
            const int live = min(16, n - 16 * q);
            if (live > 0) {
              put_HD<K>(tt, hb);
              wave_sync();
              if (n > 16 * (q + 1))
                load_tile<K>(tab, rt + 16 * (q + 1) * kRow, min(16, n - 16 * (q + 1)), 0, tt);
              else
                request(bn);
              get_chain<K>(hb, h[q], dh[q]);
              moments_tile<K, T::HD, 2>(rt + 16 * q * kRow, live, hb, acc);
              wave_sync();
            } else {
#pragma unroll
              for (int k = 0; k < T::NFB; k++) h[q][k] = dh[q][k] = 0.0f;
            }
          }
          slot_S<K>(acc, gv, g.tsym, sb);
          wave_sync();
          load_S<K>(sb, 0, so);
          wave_sync();
#pragma unroll
          for (int q = 0; q < T::RT; q++) {
            const int live = min(16, n - 16 * q);
            if (live > 0) {
              const f32x4v y = get_Y(rt + 16 * q * kRow, live);
              float f1 = 0.0f;
              f32x4v v = {0, 0, 0, 0};
              chain_block<K>(so, y, h[q], dh[q], f1, v);
              put_V(rt + 16 * q * kRow, live, f1, v);
            }
          }
          done = true;
        }
      }
      if (!done) {
        slot_moments<K>(tab, rt, n, hb, acc);
        slot_S<K>(acc, gv, g.tsym, sb);
        wave_sync();
        if constexpr (T::kSRegs) {
          load_S<K>(sb, 0, so);
          wave_sync();
        }
        slot_chain<K>(tab, rt, n, sb, so, hb);
        request(bn);
      }
      b = bn;
    }
    wave_sync();
    double cf[9];
#pragma unroll
    for (int q = 0; q < 9; q++) cf[q] = 0.0;
    if (lane < nk) neighbor_force(g, d0, (int) (e0 & kNbrJMask), rows + lane * kRow, scale, vatom, cf);
    if (64 + lane < nk) {
      double d1[3];
      displacement(xi, pos[e1 & kNbrJMask], e1 >> kNbrJBits, cell, d1);
      neighbor_force(g, d1, (int) (e1 & kNbrJMask), rows + (64 + lane) * kRow, scale, vatom, cf);
    }
    wave_sync();
    scatter<1>(rows, nk, f, vatom);
    add_sums(cf, facc);
  } else {
    force_long<K>(g, cell, xi, pos, tab, kept, start, grow, rows, hb, sb, scale, f, vatom, facc);
  }
  wave_sync();
  if (lane < 3) atomicAdd(&f[3 * (size_t) i + lane], facc[lane]);
  if (lane < 6) {
    const double v = facc[3 + lane];
    watom[6 * (size_t) i + lane] = v;
    if (vatom) atomicAdd(&vatom[6 * (size_t) i + lane], 0.5 * v);
  }
  if (lane == 6) eatom[i] = scale * E[row];
}

template <int K, int NS, bool MP>
hipError_t desc_impl(const ModelGeo &g, const Geom &geo, const double4 *pos, const uint32_t *nbr,
                     const int *nn, int cap, const int *row2atom, int rbase, int nrows, const float4 *tab,
                     float *G, uint32_t *kl, hipStream_t s)
{
  size_t offs[3];
  size_t lds = desc_lds<K>(cap, offs);
  if (lds > 160 * 1024) return hipErrorInvalidConfiguration;
  if (hipError_t ae = hipFuncSetAttribute((const void *) k_descriptor<K, NS, MP>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
      ae != hipSuccess)
    return ae;
  k_descriptor<K, NS, MP><<<nrows - rbase, 64, lds, s>>>(g, geo, pos, nbr, nn, cap, row2atom, rbase, nrows, tab,
                                                         G, kl);
  return hipGetLastError();
}

// Slots per register pass of the descriptor: the smallest of 1, 2, 4, 8 that
// holds nelt within a budget of 64 accumulators per lane; models with more
// slots than the largest such count (k = 64: 4, k = 128: 2) take several
// passes.
template <int K>
hipError_t dispatch_desc(const ModelGeo &g, const Geom &geo, const double4 *pos, const uint32_t *nbr,
                         const int *nn, int cap, const int *row2atom, int rbase, int nrows, const float4 *tab,
                         float *G, uint32_t *kl, hipStream_t s)
{
  constexpr int per = Tiling<K>::KT * 4;
  constexpr int kMaxNS = 8 * per <= 64 ? 8 : (4 * per <= 64 ? 4 : 2);
#define TMD_LAUNCH(NS, MP) \
  return desc_impl<K, NS, MP>(g, geo, pos, nbr, nn, cap, row2atom, rbase, nrows, tab, G, kl, s);
  if (g.nelt < 1 || g.nelt > kMaxElts) return hipErrorInvalidValue;
  if (g.nelt <= 1) TMD_LAUNCH(1, false)
  if (g.nelt <= 2) TMD_LAUNCH(2, false)
  if constexpr (kMaxNS >= 8) {
    if (g.nelt <= 4) TMD_LAUNCH(4, false)
    TMD_LAUNCH(8, false)
  } else if constexpr (kMaxNS == 4) {
    if (g.nelt <= 4) TMD_LAUNCH(4, false)
    TMD_LAUNCH(4, true)
  } else {
    TMD_LAUNCH(2, true)
  }
#undef TMD_LAUNCH
}

}  // namespace

hipError_t launch_descriptor(const ModelGeo &g, const Geom &geo, const double4 *pos,
                             const uint32_t *nbr, const int *nn, int cap, const int *row2atom,
                             int nrows, const float4 *tab, float *G, uint32_t *kl,
                             hipStream_t stream, int row_begin)
{
  if (nrows <= row_begin) return hipSuccess;
  if (geo.g_bf16 && g.mm > 3) return hipErrorInvalidValue;  // FP32 rows only there
  if (geo.order && row_begin != 0) return hipErrorInvalidValue;  // an order covers whole launches
  if (g.mm > 3)
    return launch_descriptor_hm(g, geo, pos, nbr, nn, cap, row2atom, nrows, tab, G, kl, stream, row_begin);
  if (!geo.dyn && desc_wide_ok(g, nrows - row_begin))
    return launch_descriptor_wide(g, geo, pos, nbr, nn, cap, row2atom, nrows, tab, G, kl, stream, row_begin);
#define TMD_K_CASE(K)                                                                                    \
  case K:                                                                                                \
    return dispatch_desc<K>(g, geo, pos, nbr, nn, cap, row2atom, row_begin, nrows, tab, G, kl, stream);
  switch (g.k) {
    TMD_K_CASE(16)
    TMD_K_CASE(24)
    TMD_K_CASE(32)
    TMD_K_CASE(64)
    TMD_K_CASE(128)
    default: return hipErrorInvalidValue;
  }
#undef TMD_K_CASE
}

hipError_t launch_force(const ModelGeo &g, const Geom &geo, const double4 *pos, int cap,
                        const int *row2atom, int nrows, const float4 *tab, const uint32_t *kl,
                        const float *dEdG, const double *E, double scale, double *f, double *eatom,
                        double *watom, double *vatom, hipStream_t stream, int row_begin)
{
  if (nrows <= row_begin) return hipSuccess;
  if (geo.order && row_begin != 0) return hipErrorInvalidValue;  // an order covers whole launches
  if (g.mm > 3)
    return launch_force_hm(g, geo, pos, cap, row2atom, nrows, tab, kl, dEdG, E, scale, f, eatom, watom, vatom,
                           stream, row_begin);
  if (!geo.dyn && force_waves(g, nrows - row_begin) > 1)
    return launch_force_wide(g, geo, pos, cap, row2atom, nrows, tab, kl, dEdG, E, scale, f, eatom, watom, vatom,
                             stream, row_begin);
#define TMD_K_CASE(K)                                                                                       \
  case K:                                                                                                   \
    k_force<K><<<nrows - row_begin, 64, 0, stream>>>(g, geo, pos, cap, row2atom, row_begin, nrows, tab, kl, \
                                                     dEdG, E, scale, f, eatom, watom, vatom);               \
    return hipGetLastError();
  switch (g.k) {
    TMD_K_CASE(16)
    TMD_K_CASE(24)
    TMD_K_CASE(32)
    TMD_K_CASE(64)
    TMD_K_CASE(128)
    default: return hipErrorInvalidValue;
  }
#undef TMD_K_CASE
}

}  // namespace tmd
