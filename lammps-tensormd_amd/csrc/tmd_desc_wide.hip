// Descriptor and force kernels with several waves per atom, for small systems
// (gfx950, wave64, max_moment 0-3, at most 32 filters): the method and the
// operand layouts are those of tmd_desc.hip.
//
// In a file of their own: compiled beside the one-wave kernels they cost the
// latter's registers (k_force<24> then spilled 3, and 128,000 atoms took 653
// instead of 619 us).
#include "tmd_desc_moments.h"

#include <algorithm>

namespace tmd {

namespace {

// ---- several waves per atom ----
// A small system gives a CU few waves, and a wave's chain of loads, tiles and
// reductions is then all latency.  W waves share an atom: a lane takes one
// list entry and, while its geometry is in registers, stages it; the tiles
// of neighbors are dealt out to the waves, and their P are added in a fixed
// order.  Lists or kept counts beyond the workgroup's room are left to its
// first wave.  (Figures at force_waves.)
constexpr int kWideRows = 96;  // staged neighbors of the descriptor
constexpr int kDescWaves = 4;

template <int K, int NS>
struct DescWide {
  float rows[kWideRows * kRow];
  float hb[kDescWaves][Tiling<K>::HBUF];
  f32x4v part[kDescWaves][NS * Tiling<K>::KT][64];
  int cnt[kMaxElts][kDescWaves];
};

template <int K, int NS>
__global__ __launch_bounds__(64 * kDescWaves) void k_descriptor_wide(ModelGeo g, Geom geo, const double4 *pos,
                                                                const uint32_t *nbr, const int *nn, int cap,
                                                                const int *row2atom, int rbase, int nrows,
                                                                const float4 *tab, float *G, uint32_t *kl)
{
  using T = Tiling<K>;
  extern __shared__ __align__(16) unsigned char smem[];
  const int row = geo.order ? geo.order[rbase + (int) blockIdx.x] : rbase + (int) blockIdx.x;
  if (row >= nrows) return;
  float *Grow;
  const int i = descriptor_begin(g, geo, K, row, row2atom, G, Grow);
  if (i < 0) return;
  DescWide<K, NS> &sh = *reinterpret_cast<DescWide<K, NS> *>(smem);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nraw = nn[i];
  if (nraw <= 64 * kDescWaves) {
    const uint32_t *list = nbr + (size_t) i * cap;
    const uint32_t le = list[min(tid, max(nraw - 1, 0))];
    const uint32_t e = tid < nraw ? le : 0u;
    const double4 xi = pos[i];
    const Box cell = load_box(geo, i);
    NbrGeo ng;
    const int sl = kept_slot(g, cell, xi, (int) xi.w, e, pos[e & kNbrJMask], ng.d);
    const int slot = tid < nraw ? sl : -1;
    int rank = 0;
    for (int b = 0; b < g.nelt; b++) {
      const unsigned long long m = __ballot(slot == b);
      if (slot == b) rank = (int) lane_rank(m);
      if (lane == 0) sh.cnt[b][wave] = __popcll(m);
    }
    __syncthreads();
    int start[NS + 1], nk = 0;
#pragma unroll
    for (int b = 0; b < NS; b++) {
      start[b] = nk;
      if (b < g.nelt) {
#pragma unroll
        for (int w = 0; w < kDescWaves; w++) {
          if (slot == b && w < wave) rank += sh.cnt[b][w];
          nk += sh.cnt[b][w];
        }
        if (slot == b) rank += start[b];
      }
    }
    start[NS] = nk;
    if (nk <= kWideRows) {
      uint32_t *kr = kl + (size_t) row * kept_cache_words(cap);
      if (slot >= 0) {
        kr[kKeptHdr + rank] = e;
        nbr_geometry(g, ng);
        put_row(ng, sh.rows + rank * kRow);
      }
      if (tid == 0) {
        kr[0] = (uint32_t) nk;
#pragma unroll
        for (int b = 0; b <= NS; b++)
          if (b <= g.nelt) kr[1 + b] = (uint32_t) start[b];
      }
      __syncthreads();
      f32x4v acc[NS][T::KT];
#pragma unroll
      for (int b = 0; b < NS; b++)
#pragma unroll
        for (int t = 0; t < T::KT; t++) acc[b][t] = f32x4v{0, 0, 0, 0};
      for (int r0 = 16 * wave; r0 < nk; r0 += 16 * kDescWaves) {
        TabTile<K> tt;
        load_tile<K>(tab, sh.rows + r0 * kRow, min(16, nk - r0), 0, tt);
        descriptor_tile<K, NS>(tt, [] {}, sh.rows + r0 * kRow, r0, min(16, nk - r0), 0, start, g.nelt, sh.hb[wave], acc);
        wave_sync();
      }
#pragma unroll
      for (int b = 0; b < NS; b++)
#pragma unroll
        for (int t = 0; t < T::KT; t++) sh.part[wave][b * T::KT + t][lane] = acc[b][t];
      __syncthreads();
      for (int p = wave; p < g.nelt * T::KT; p += kDescWaves) {
        f32x4v v = sh.part[0][p][lane];
#pragma unroll
        for (int w = 1; w < kDescWaves; w++) v += sh.part[w][p][lane];
        store_g<K>(v, p / T::KT, p % T::KT, g.tsym, Grow, geo.g_bf16);
      }
      return;
    }
    __syncthreads();
  }
  if (wave == 0) descriptor_row<K, NS, false>(g, geo, row, i, pos, nbr, nn, cap, tab, Grow, kl, smem);
}

// W waves per atom (as k_descriptor_wide): one neighbor per lane, and the
// slots dealt out to the waves; with one or two slots, four or two waves
// share the tiles of a slot and add their P in a fixed order.
template <int K, int W, int SHARE>
__global__ __launch_bounds__(64 * W, (K <= 16 ? 4 : 3)) void k_force_wide(ModelGeo g, Geom geo, const double4 *pos, int cap,
                                              const int *row2atom, int rbase, int nrows, const float4 *tab,
                                              const uint32_t *kl, const float *dEdG,
                                              const double *E, double scale, double *f,
                                              double *eatom, double *watom, double *vatom)
{
  using T = Tiling<K>;
  static_assert(T::kSRegs && T::NB == 1 && T::WIN <= 128, "S in registers, one block, two waves of neighbors");
  // tiles of a slot whose H and dH a wave holds: a window over the waves that
  // share it, two of a slot that is not shared
  constexpr int QT = SHARE == 1 ? 2 : ((T::WIN + 15) / 16 + SHARE - 1) / SHARE;
  __shared__ __align__(16) float rows[T::WIN * kRow];
  __shared__ __align__(16) float buf[W][T::BUF];
  __shared__ __align__(16) f32x4v part[SHARE > 1 ? W : 1][T::KT][64];
  __shared__ double facc[2][9];
  const int row = geo.order ? geo.order[rbase + (int) blockIdx.x] : rbase + (int) blockIdx.x;
  if (row >= nrows) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = row2atom[row];
  if (i < 0) return;  // padding row
  float *hb = buf[wave];
  const double4 xi = pos[i];
  const Box cell = load_box(geo, i);
  const uint32_t *kr = kl + (size_t) row * kept_cache_words(cap);
  const uint32_t *kept = kr + kKeptHdr;
  const uint32_t hdr = kr[lane & 15];
  const uint32_t e = kept[min(tid, cap - 1)];
  const int nk = (int) __builtin_amdgcn_readlane((int) hdr, 0);
  auto start = [&](int b) { return (int) __builtin_amdgcn_readlane((int) hdr, 1 + b); };
  const float *grow = dEdG + (size_t) row * g.nelt * K * kNM;
  if (tid < 18) facc[tid / 9][tid % 9] = 0.0;
  if (nk <= T::WIN) {
    double d[3] = {0.0, 0.0, 0.0};
    if (tid < nk) stage_row(g, cell, xi, pos, e, rows + tid * kRow, d);
    __syncthreads();
    const int first = wave % SHARE;
    // with shared slots every wave takes one slot: all reach the barrier
    for (int b = wave / SHARE; b < g.nelt; b += W / SHARE) {
      const int s0 = start(b), n = start(b + 1) - s0;
      if (SHARE == 1 && n == 0) continue;
      float *rt = rows + s0 * kRow;
      float4 gv[T::KT];
      load_dEdG<K>(grow + (size_t) b * K * kNM, gv);
      f32x4v acc[T::KT];
#pragma unroll
      for (int t = 0; t < T::KT; t++) acc[t] = f32x4v{0, 0, 0, 0};
      SOps<K> so;
      if (n <= 16 * QT * SHARE) {
        auto live = [&](int q) { return min(16, n - 16 * (first + q * SHARE)); };
        auto tile = [&](int q) { return rt + 16 * (first + q * SHARE) * kRow; };
        float h[QT][T::NFB], dh[QT][T::NFB];
        TabTile<K> tt;
        if (live(0) > 0) load_tile<K>(tab, tile(0), live(0), 0, tt);
#pragma unroll
        for (int q = 0; q < QT; q++) {
          if (live(q) > 0) {
            put_HD<K>(tt, hb);
            wave_sync();
            if (q + 1 < QT && live(q + 1) > 0) load_tile<K>(tab, tile(q + 1), live(q + 1), 0, tt);
            get_chain<K>(hb, h[q], dh[q]);
            moments_tile<K, T::HD, 2>(tile(q), live(q), hb, acc);
            wave_sync();
          } else {
#pragma unroll
            for (int k = 0; k < T::NFB; k++) h[q][k] = dh[q][k] = 0.0f;
          }
        }
        if constexpr (SHARE > 1) {
#pragma unroll
          for (int t = 0; t < T::KT; t++) part[wave][t][lane] = acc[t];
          __syncthreads();
#pragma unroll
          for (int t = 0; t < T::KT; t++) {
            acc[t] = part[wave - first][t][lane];
            for (int w = 1; w < SHARE; w++) acc[t] += part[wave - first + w][t][lane];
          }
        }
        if (live(0) > 0) {
          slot_S<K>(acc, gv, g.tsym, hb);
          wave_sync();
          load_S<K>(hb, 0, so);
          wave_sync();
#pragma unroll
          for (int q = 0; q < QT; q++) {
            if (live(q) > 0) {
              const f32x4v y = get_Y(tile(q), live(q));
              float f1 = 0.0f;
              f32x4v v = {0, 0, 0, 0};
              chain_block<K>(so, y, h[q], dh[q], f1, v);
              put_V(tile(q), live(q), f1, v);
            }
          }
        }
      } else if constexpr (SHARE == 1) {
        slot_moments<K>(tab, rt, n, hb, acc);
        slot_S<K>(acc, gv, g.tsym, hb);
        wave_sync();
        load_S<K>(hb, 0, so);
        wave_sync();
        slot_chain<K>(tab, rt, n, hb, so, hb);
      }
    }
    __syncthreads();
    if (wave < 2) {
      double cf[9];
#pragma unroll
      for (int q = 0; q < 9; q++) cf[q] = 0.0;
      if (tid < nk) neighbor_force(g, d, (int) (e & kNbrJMask), rows + tid * kRow, scale, vatom, cf);
      add_sums(cf, facc[wave]);
    }
    __syncthreads();
    scatter<W>(rows, nk, f, vatom);
  } else {
    __syncthreads();
    if (wave == 0)
      force_long<K>(g, cell, xi, pos, tab, kept, start, grow, rows, hb, hb, scale, f, vatom, facc[0]);
  }
  if (wave != 0) return;
  wave_sync();
  if (lane < 3) atomicAdd(&f[3 * (size_t) i + lane], facc[0][lane] + facc[1][lane]);
  if (lane < 6) {
    const double v = facc[0][3 + lane] + facc[1][3 + lane];
    watom[6 * (size_t) i + lane] = v;
    if (vatom) atomicAdd(&vatom[6 * (size_t) i + lane], 0.5 * v);
  }
  if (lane == 6) eatom[i] = scale * E[row];
}

template <int K, int W>
hipError_t force_wide(const ModelGeo &g, const Geom &geo, const double4 *pos, int cap, const int *row2atom, int rbase,
                      int nrows, const float4 *tab, const uint32_t *kl, const float *dEdG, const double *E,
                      double scale, double *f, double *eatom, double *watom, double *vatom, hipStream_t s)
{
  auto go = [&](auto kern) {
    kern<<<nrows - rbase, 64 * W, 0, s>>>(g, geo, pos, cap, row2atom, rbase, nrows, tab, kl, dEdG, E, scale, f,
                                              eatom, watom, vatom);
    return hipGetLastError();
  };
  return g.nelt == 1 ? go(k_force_wide<K, W, W>) : (g.nelt == 2 ? go(k_force_wide<K, W, W / 2>) : go(k_force_wide<K, W, 1>));
}

// slots accumulated by the descriptor kernel
constexpr int desc_slots(int nelt) { return nelt <= 1 ? 1 : (nelt <= 2 ? 2 : (nelt <= 4 ? 4 : 8)); }

template <int K, int NS>
hipError_t desc_wide(const ModelGeo &g, const Geom &geo, const double4 *pos, const uint32_t *nbr, const int *nn, int cap,
                     const int *row2atom, int rbase, int nrows, const float4 *tab, float *G, uint32_t *kl, hipStream_t s)
{
  if constexpr (NS * Tiling<K>::KT <= 8) {
    size_t offs[3];
    const size_t lds = std::max(desc_lds<K>(cap, offs), sizeof(DescWide<K, NS>));
    if (lds > 160 * 1024) return hipErrorInvalidConfiguration;
    if (hipError_t ae = hipFuncSetAttribute((const void *) k_descriptor_wide<K, NS>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
        ae != hipSuccess)
      return ae;
    k_descriptor_wide<K, NS><<<nrows - rbase, 64 * kDescWaves, lds, s>>>(g, geo, pos, nbr, nn, cap, row2atom, rbase, nrows,
                                                                   tab, G, kl);
    return hipGetLastError();
  } else {
    return hipErrorInvalidValue;
  }
}

}  // namespace

// Waves per atom (K <= 32).  Several shorten a wave's chain but add barriers
// and, in the lane-per-neighbor parts, idle lanes, so they pay while a CU has
// few atoms.  (The descriptor's two-wave form won 1 us in a narrow band and
// is not built.)  us, descriptor with 1 and 4 waves, force with 1, 2 and 4:
//   elements, K   rows   descriptor        force
//     1, 16        512   10.2   7.9   14.7  13.5  12.8
//                1,408   11.7  11.0   17.1  16.3  18.6
//                2,048   12.1  12.4   20.0  18.1  21.7
//                2,944   13.6  15.3   23.9  25.5  27.1
//     1, 24      1,024    9.7   9.0   15.4  13.6  13.5
//                2,048   11.1  12.9   20.4  20.7  20.9
//     1, 32        704    9.7   8.5   15.8  13.4  12.6
//                2,048   11.4  13.4   22.5  20.7  23.8
//                3,456   14.5  19.3   28.4  28.5  33.3
//     2, 32        512   10.0   8.4   15.9  13.7  11.9
//                1,408   11.4  12.4   19.8  16.7  18.5
//                2,944   14.1  18.8   26.3  25.3  29.2
//     3, 16        576    9.6   8.4   14.4  13.0  12.2
//                1,536   10.9  12.6   19.3  18.1  18.8
//                2,688   12.4  17.7   21.8  23.8  24.5
//     4, 24        512   10.7   9.2   15.9  13.7  12.4
//                  768   10.8   9.8   16.1  13.9  12.9
//                1,024   11.1  13.0   16.4  14.6  17.8
//                1,536   12.2  14.9   21.6  18.4  20.9
//                2,048   12.7  18.8   21.5  23.3  25.9
//     5, 24        640                 16.6  14.2  12.8
//                1,600                 22.8  20.1  21.9
//                2,240                 23.4  25.8  28.4
//     8, 32        512                 20.9  15.3  13.2
//                2,048                 30.8  28.4  28.7
constexpr int kWide4Rows = 640, kWide2Rows = 1600;

int force_waves(const ModelGeo &g, int rows)
{
  if (g.k > 32) return 1;
  if (rows <= kWide4Rows) return 4;
  return rows <= (g.nelt <= 2 ? 2048 : kWide2Rows) ? 2 : 1;
}

// the sums of the waves' P fit beside four workgroups' others up to 8 filter
// tiles
bool desc_wide_ok(const ModelGeo &g, int rows)
{
  return g.k <= 32 && desc_slots(g.nelt) * ((g.k + 15) / 16) <= 8 && rows <= kWide4Rows;
}

hipError_t launch_descriptor_wide(const ModelGeo &g, const Geom &geo, const double4 *pos, const uint32_t *nbr,
                                  const int *nn, int cap, const int *row2atom, int nrows, const float4 *tab, float *G,
                                  uint32_t *kl, hipStream_t s, int row_begin)
{
  if (geo.dyn || !desc_wide_ok(g, nrows - row_begin) || g.nelt < 1 || g.nelt > kMaxElts) return hipErrorInvalidValue;
#define TMD_NS(K, NS) \
  case NS:            \
    return desc_wide<K, NS>(g, geo, pos, nbr, nn, cap, row2atom, row_begin, nrows, tab, G, kl, s);
#define TMD_K_CASE(K)              \
  case K:                          \
    switch (desc_slots(g.nelt)) {  \
      TMD_NS(K, 1)                 \
      TMD_NS(K, 2)                 \
      TMD_NS(K, 4)                 \
      TMD_NS(K, 8)                 \
    }                              \
    return hipErrorInvalidValue;
  switch (g.k) {
    TMD_K_CASE(16)
    TMD_K_CASE(24)
    TMD_K_CASE(32)
    default: return hipErrorInvalidValue;
  }
#undef TMD_K_CASE
#undef TMD_NS
}

hipError_t launch_force_wide(const ModelGeo &g, const Geom &geo, const double4 *pos, int cap, const int *row2atom,
                             int nrows, const float4 *tab, const uint32_t *kl, const float *dEdG, const double *E,
                             double scale, double *f, double *eatom, double *watom, double *vatom, hipStream_t s,
                             int row_begin)
{
  const int w = force_waves(g, nrows - row_begin);
  if (geo.dyn || w <= 1) return hipErrorInvalidValue;
#define TMD_K_CASE(K)                                                                                               \
  case K:                                                                                                           \
    return w == 4 ? force_wide<K, 4>(g, geo, pos, cap, row2atom, row_begin, nrows, tab, kl, dEdG, E, scale, f,      \
                                     eatom, watom, vatom, s)                                                        \
                  : force_wide<K, 2>(g, geo, pos, cap, row2atom, row_begin, nrows, tab, kl, dEdG, E, scale, f,      \
                                     eatom, watom, vatom, s);
  switch (g.k) {
    TMD_K_CASE(16)
    TMD_K_CASE(24)
    TMD_K_CASE(32)
    default: return hipErrorInvalidValue;
  }
#undef TMD_K_CASE
}

}  // namespace tmd
