// The moment kernels' parts for max_moment 0-3, shared by the kernels with one
// wave per atom (tmd_desc.hip, where the method is described) and with several
// (tmd_desc_wide.hip).
#pragma once
#include "tmd_desc_common.h"

namespace tmd {

namespace {

typedef float f32x4v __attribute__((ext_vector_type(4)));

constexpr int kNY = 16;  // harmonics of degree 0..3: degree l starts at l^2
// LDS row of a staged neighbor: 16 harmonics, then q, 1 - q and the table
// cell.  A stride of 20 words puts the 16-byte accesses of 16 rows on
// distinct banks.
constexpr int kRow = 20;

// Filters are taken in blocks of FBL (all of them up to K = 32, else 32).
template <int K>
struct Tiling {
  static constexpr int FBL = K <= 32 ? K : 32;
  static constexpr int NFB = FBL / 4;          // filters of a block per lane
  static constexpr int NB = K / FBL;           // blocks
  static constexpr int CT = (FBL + 15) / 16;   // filter tiles per block
  static constexpr int KT = NB * CT;           // filter tiles
  // the second tile of K = 24 holds 8 filters, the others 16
  static constexpr int nper(int t) { return (K == 24 && t == 1) ? 2 : 4; }  // filters per lane group
  // H of 16 neighbors, [16][HS], and H with dH interleaved, [16][HD]: HS / 4
  // and HD / 4 are odd, so the quads of 16 rows hit distinct banks
  static constexpr int HS = FBL + 4, HD = 2 * FBL + 4;
  static constexpr int SS = kRow;              // stride of an S row
  // S is kept in registers per slot up to K = 32, and its LDS then overlays H
  static constexpr bool kSRegs = K <= 32;
  // floats (the second tile of K = 24 reads 4 or 12 past row 15)
  static constexpr int HBUF = 16 * HS + 4, DBUF = 16 * HD + (K == 24 ? 12 : 0);
  static constexpr int SBUF = K * SS;
  static constexpr int BUF = kSRegs ? (DBUF > SBUF ? DBUF : SBUF) : DBUF + SBUF;
  // staged neighbors of the force kernel: what leaves 16 waves per CU
  // (10 KB each) up to K = 32; above, one per lane (a CU holds 11 and 8 waves
  // of K = 64 and 128).  A longer list goes slot by slot, at no step in time:
  // K = 64, 35,152 atoms, 291 us with 56 neighbors and 296 with 75.
  static constexpr int WIN = K == 16 ? 96 : (K == 24 ? 84 : (K == 32 ? 72 : 64));
  // tiles of a slot whose H and dH stay in registers between P and the
  // chain rule (2 NFB registers each)
  static constexpr int RT = K == 16 ? 5 : (K <= 32 ? 2 : 0);
};

// Y_d(u) in d order: 1 | x y z | 5 of degree 2 | 7 of degree 3, scaled so
// that the sums of squares above hold.
__device__ inline void harmonics(float x, float y, float z, float *Y)
{
  constexpr float r2 = 1.4142135623730951f, r6 = 2.4494897427831781f;
  const float zz = z * z, xy = x * y, xxyy = (x - y) * (x + y);
  Y[0] = 1.0f;
  Y[1] = x;
  Y[2] = y;
  Y[3] = z;
  Y[4] = fmaf(1.2247448713915890f, zz, -0.40824829046386302f);  // (3 z^2 - 1) / sqrt 6
  Y[5] = r2 * x * z;
  Y[6] = r2 * y * z;
  Y[7] = 0.70710678118654752f * xxyy;
  Y[8] = r2 * xy;
  Y[9] = z * fmaf(1.5811388300841898f, zz, -0.94868329805051381f);  // z (5 z^2 - 3) / sqrt 10
  const float p = fmaf(1.9364916731037085f, zz, -0.38729833462074170f);  // sqrt(3/20) (5 z^2 - 1)
  Y[10] = p * x;
  Y[11] = p * y;
  Y[12] = 0.5f * r6 * z * xxyy;
  Y[13] = r6 * xy * z;
  Y[14] = 0.5f * x * fmaf(x, x, -3.0f * y * y);
  Y[15] = 0.5f * y * fmaf(3.0f * x, x, -y * y);
}

// g = sum_d V_d dY_d/du (the polynomials above as functions of a free u)
__device__ inline void harmonics_grad(float x, float y, float z, const float *V, float &gx, float &gy, float &gz)
{
  constexpr float r2 = 1.4142135623730951f, r6 = 2.4494897427831781f, a10 = 3.8729833462074170f;
  const float zz = z * z, xxyy = (x - y) * (x + y);
  const float p = fmaf(1.9364916731037085f, zz, -0.38729833462074170f);
  const float x2 = r2 * x, y2 = r2 * y, z2 = r2 * z, x6 = r6 * x, y6 = r6 * y, z6 = r6 * z;
  const float d14 = 1.5f * xxyy, xy3 = 3.0f * x * y;
  gx = V[1] + z2 * V[5] + x2 * V[7] + y2 * V[8] + p * V[10] + x6 * z * V[12] + y6 * z * V[13] + d14 * V[14] +
      xy3 * V[15];
  gy = V[2] + z2 * V[6] - y2 * V[7] + x2 * V[8] + p * V[11] - y6 * z * V[12] + x6 * z * V[13] - xy3 * V[14] +
      d14 * V[15];
  gz = V[3] + z6 * V[4] + x2 * V[5] + y2 * V[6] + fmaf(4.7434164902525694f, zz, -0.94868329805051381f) * V[9] +
      a10 * z * (x * V[10] + y * V[11]) + 0.5f * r6 * xxyy * V[12] + x6 * y * V[13];
}

// The LDS row of a neighbor.
__device__ inline void put_row(const NbrGeo &ng, float *rowp)
{
  float Y[kNY];
  harmonics(ng.ux, ng.uy, ng.uz, Y);
  float4 *r = reinterpret_cast<float4 *>(rowp);
#pragma unroll
  for (int q = 0; q < 4; q++) r[q] = make_float4(Y[4 * q], Y[4 * q + 1], Y[4 * q + 2], Y[4 * q + 3]);
  // a table of one point has no cell: its only row is an end row
  r[4] = make_float4(ng.q, ng.pq, __int_as_float(max(ng.n, 0)), 0.0f);
}

// The LDS row of neighbor e; d receives its displacement.
__device__ inline void stage_row(const ModelGeo &g, const Box &cell, const double4 &xi, const double4 *pos,
                                 uint32_t e, float *rowp, double d[3])
{
  NbrGeo ng;
  nbr_geometry(g, cell, xi, pos, e, ng);
  put_row(ng, rowp);
#pragma unroll
  for (int q = 0; q < 3; q++) d[q] = ng.d[q];
}

// rows[c] of the n entries list[0..n)
__device__ inline void stage(const ModelGeo &g, const Box &cell, const double4 &xi, const double4 *pos,
                             const uint32_t *list, int n, float *rows)
{
  for (int c = threadIdx.x & 63; c < n; c += 64) {
    double d[3];
    stage_row(g, cell, xi, pos, list[c], rows + c * kRow, d);
  }
  wave_sync();
}

// The table rows of one block of filters for the tile of neighbors
// rows[0..live), live >= 1: lane l takes the filters 4 i + l % 4 of neighbor
// l / 4, so that 4 lanes read 64 contiguous bytes.  The table's end cells are
// zero rows, and a lane past the tile takes row 0: H = dH = 0 there without
// a mask.
template <int K>
struct TabTile {
  float4 t[Tiling<K>::NFB];
  float q, pq;
};

template <int K>
__device__ inline void load_tile(const float4 *tab, const float *rows, int live, int block, TabTile<K> &o)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63, c = lane >> 2;
  const float4 v = *reinterpret_cast<const float4 *>(rows + min(c, live - 1) * kRow + kNY);
  const int n = c < live ? __float_as_int(v.z) : 0;
  o.q = v.x;
  o.pq = v.y;
  const float4 *row = tab + (size_t) n * K + block * T::FBL + (lane & 3);
#pragma unroll
  for (int i = 0; i < T::NFB; i++) o.t[i] = row[4 * i];
}

// a block's H of the tile -> hb [16][HS]
template <int K>
__device__ inline void put_H(const TabTile<K> &o, float *hb)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63;
  float *p = hb + (lane >> 2) * T::HS + (lane & 3);
#pragma unroll
  for (int i = 0; i < T::NFB; i++) p[4 * i] = kerley_h(o.t[i], o.q, o.pq);
}

// a block's H and dH = dx H' of the tile -> hb [16][HD]
template <int K>
__device__ inline void put_HD(const TabTile<K> &o, float *hb)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63;
  float *p = hb + (lane >> 2) * T::HD + 2 * (lane & 3);
#pragma unroll
  for (int i = 0; i < T::NFB; i++) {
    float2 v;
    kerley(o.t[i], o.q, o.pq, o.q - o.pq, v.x, v.y);
    *reinterpret_cast<float2 *>(p + 8 * i) = v;
  }
}

// H and dH of neighbor l % 16 in the chain-rule layout: lane group l / 16
// holds nper(t) consecutive filters of tile t
template <int K>
__device__ inline void get_chain(const float *hb, float *h, float *dh)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63, grp = lane >> 4;
  const float *p = hb + (lane & 15) * T::HD;
#pragma unroll
  for (int t = 0; t < T::CT; t++) {
    const int np = T::nper(t);
#pragma unroll
    for (int i = 0; i < np; i += 2) {
      const float4 v = *reinterpret_cast<const float4 *>(p + 2 * (16 * t + np * grp + i));
      h[4 * t + i] = v.x;
      dh[4 * t + i] = v.y;
      h[4 * t + i + 1] = v.z;
      dh[4 * t + i + 1] = v.w;
    }
  }
}

// P of a block's filters += the tile in rows[0..live): P^T[d][k] of tile t
// in acc[t].  Filter k of neighbor c is hb[c STR + k SK]; rows past the tile
// hold H = 0.
template <int K, int STR, int SK>
__device__ inline void moments_tile(const float *rows, int live, const float *hb, f32x4v *acc)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63;
  float a[4], b[4][T::CT];
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int c = 4 * s + (lane >> 4);
    a[s] = rows[min(c, live - 1) * kRow + (lane & 15)];
#pragma unroll
    for (int t = 0; t < T::CT; t++) b[s][t] = hb[c * STR + SK * (16 * t + (lane & 15))];
  }
#pragma unroll
  for (int s = 0; s < 4; s++) {
    if (4 * s >= live) break;
#pragma unroll
    for (int t = 0; t < T::CT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s][t], acc[t], 0, 0, 0);
  }
}

// G[b][k][0..3] of one filter tile from its P^T: lane group m ends up with
// component m of filter l % 16 (fixed-order sums over the groups).
__device__ inline float g_components(const f32x4v &p, int tsym)
{
  const int grp = (threadIdx.x & 63) >> 4;
  const float a = p[0] * p[0], b = p[1] * p[1] + p[2] * p[2] + p[3] * p[3];
  const float c2 = tsym ? 0.0f : (1.0f / 3.0f), c3 = tsym ? 0.0f : 0.6f;
  // degrees of a group's harmonics: 0 111 | 2222 | 2 333 | 3333
  const float t0 = grp == 0 ? p[0] : 0.0f;
  const float t1 = grp == 0 ? b : 0.0f;
  const float t2 = (grp == 0 ? c2 : (grp == 3 ? 0.0f : 1.0f)) * a + (grp == 1 ? 1.0f : 0.0f) * b;
  const float t3 = (grp == 3 ? 1.0f : 0.0f) * a + (grp == 0 ? c3 : (grp == 1 ? 0.0f : 1.0f)) * b;
  return swap16_add(swap32_add(t0, t2), swap32_add(t1, t3));
}

// descriptor LDS: kept list and staged rows, or the rows of all kept
// neighbors; H
constexpr int kDescWin = 64, kDescAll = 88;
template <int K>
__host__ __device__ inline size_t desc_lds(int cap, size_t *offs)
{
  size_t o = 0;
  auto take = [&](size_t bytes) {
    size_t r = o;
    o += (bytes + 15) & ~(size_t) 15;
    return r;
  };
  offs[0] = take((size_t) cap * 4);
  offs[1] = take((size_t) kDescWin * kRow * 4);
  o = o > kDescAll * kRow * 4 ? o : kDescAll * kRow * 4;
  offs[2] = take((size_t) Tiling<K>::HBUF * 4);
  return o;
}

// P of the nsl slots of one pass (kept entries start[0] .. start[nsl], slot
// sorted) += the tile of `live` neighbors from entry `first` on, staged in
// rt.  Tiles run across slot boundaries: each slot takes its own neighbors
// of a tile by zeroing the harmonics of the others.
template <int K, int NS, typename Next>
__device__ inline void descriptor_tile(TabTile<K> &tt, const Next &next, const float *rt, int first, int live, int fb,
                                       const int *start, int nsl, float *hb, f32x4v (&acc)[NS][Tiling<K>::KT])
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63;
  put_H<K>(tt, hb);
  wave_sync();
  next();
  float a[4], bo[4][T::CT];
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int c = 4 * s + (lane >> 4);
    a[s] = rt[min(c, live - 1) * kRow + (lane & 15)];
#pragma unroll
    for (int t = 0; t < T::CT; t++) bo[s][t] = hb[c * T::HS + 16 * t + (lane & 15)];
  }
#pragma unroll
  for (int b = 0; b < NS; b++) {
    if (b >= nsl) break;
    const int lo = max(start[b] - first, 0), hi = min(start[b + 1] - first, live);
    if (lo >= hi) continue;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      if (4 * s >= hi || 4 * s + 4 <= lo) continue;
      const int c = 4 * s + (lane >> 4);
      const float as = (c >= lo && c < hi) ? a[s] : 0.0f;
#pragma unroll
      for (int t = 0; t < T::CT; t++)
        acc[b][fb * T::CT + t] =
            __builtin_amdgcn_mfma_f32_16x16x4f32(as, bo[s][t], acc[b][fb * T::CT + t], 0, 0, 0);
    }
  }
}

// The descriptor row's values of slot b, filter tile t from P^T.
template <int K>
__device__ inline void store_g(const f32x4v &p, int b, int t, int tsym, float *Grow, bool gbf16)
{
  const int lane = threadIdx.x & 63;
  const float v = g_components(p, tsym);
  const int k = 16 * t + (lane & 15);
  if (k < K) {
    const size_t o = ((size_t) b * K + k) * kNM + (lane >> 4);
    if (gbf16)
      reinterpret_cast<__bf16 *>(Grow)[o] = (__bf16) v;
    else
      Grow[o] = v;
  }
}

// P of the nsl slots of one pass over the kept entries kept[start[0],
// start[nsl]) (slot-sorted), then G.
template <int K, int NS>
__device__ inline void descriptor_pass(const ModelGeo &g, const Box &cell, const double4 &xi, const double4 *pos,
                                       const float4 *tab, const uint32_t *kept, const int *start, int nsl,
                                       float *rows, float *hb, float *Grow, int b0, bool gbf16, bool staged = false)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63;
  f32x4v acc[NS][T::KT];
#pragma unroll
  for (int b = 0; b < NS; b++)
#pragma unroll
    for (int t = 0; t < T::KT; t++) acc[b][t] = f32x4v{0, 0, 0, 0};
  const int end = start[nsl];
  const int win = staged ? end : kDescWin;
  for (int w0 = start[0]; w0 < end; w0 += win) {
    const int nw = min(win, end - w0);
    if (!staged) stage(g, cell, xi, pos, kept + w0, nw, rows);
    TabTile<K> tt;
    load_tile<K>(tab, rows, min(16, nw), 0, tt);
    for (int r0 = 0; r0 < nw; r0 += 16) {
      const int live = min(16, nw - r0);
      const float *rt = rows + r0 * kRow;
#pragma unroll
      for (int fb = 0; fb < T::NB; fb++) {
        auto next = [&]() {
          const int r = fb + 1 < T::NB ? r0 : r0 + 16;
          if (r < nw) load_tile<K>(tab, rows + r * kRow, min(16, nw - r), (fb + 1) % T::NB, tt);
        };
        descriptor_tile<K, NS>(tt, next, rt, w0 + r0, live, fb, start, nsl, hb, acc);
        wave_sync();
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NS; b++) {
    if (b >= nsl) break;
#pragma unroll
    for (int t = 0; t < T::KT; t++) {
      store_g<K>(acc[b][t], b0 + b, t, g.tsym, Grow, gbf16);
    }
  }
}

// The row of atom i by one wave.  NS: slots accumulated per register pass.
// MP: the model has more slots than NS, and the wave runs ceil(nelt / NS)
// passes over the slot-sorted kept list (each neighbor is still staged once).
template <int K, int NS, bool MP>
__device__ inline void descriptor_row(const ModelGeo &g, const Geom &geo, int row, int i, const double4 *pos,
                                      const uint32_t *nbr, const int *nn, int cap, const float4 *tab, float *Grow,
                                      uint32_t *kl, unsigned char *smem)
{
  const int lane = threadIdx.x & 63;
  size_t offs[3];
  desc_lds<K>(cap, offs);
  uint32_t *kept = reinterpret_cast<uint32_t *>(smem + offs[0]);
  float *rows = reinterpret_cast<float *>(smem + offs[1]);
  float *hb = reinterpret_cast<float *>(smem + offs[2]);
  float *all = reinterpret_cast<float *>(smem);  // kDescAll rows, over the kept list and the window
  int start[kMaxElts + 1];
  const double4 xi = pos[i];
  const Box cell = load_box(geo, i);
  uint32_t *kr = kl + (size_t) row * kept_cache_words(cap);
  if constexpr (!MP) {
    // a list of at most two entries per lane: their geometry stays in
    // registers, and the kept ones are staged from there instead of being
    // gathered and displaced a second time (128,000 atoms, with the table rows
    // of the next tile requested ahead: 334 -> 302 us)
    const int nraw = nn[i];
    if (nraw <= 128) {
      const uint32_t *list = nbr + (size_t) i * cap;
      const int last = max(nraw - 1, 0);
      uint32_t ent[2];
      double4 xj[2];
      NbrGeo ng[2];
      int slot[2], rank[2] = {0, 0};
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const uint32_t e = list[min(64 * c + lane, last)];
        ent[c] = 64 * c + lane < nraw ? e : 0u;
      }
#pragma unroll
      for (int c = 0; c < 2; c++) xj[c] = pos[ent[c] & kNbrJMask];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const int sl = kept_slot(g, cell, xi, (int) xi.w, ent[c], xj[c], ng[c].d);
        slot[c] = 64 * c + lane < nraw ? sl : -1;
      }
      int nk = 0;
      for (int b = 0; b < g.nelt; b++) {
        start[b] = nk;
#pragma unroll
        for (int c = 0; c < 2; c++) {
          const unsigned long long m = __ballot(slot[c] == b);
          if (slot[c] == b) rank[c] = nk + (int) lane_rank(m);
          nk += __popcll(m);
        }
      }
      start[g.nelt] = nk;
      if (nk <= kDescAll) {
#pragma unroll
        for (int c = 0; c < 2; c++)
          if (slot[c] >= 0) {
            kr[kKeptHdr + rank[c]] = ent[c];
            nbr_geometry(g, ng[c]);
            put_row(ng[c], all + rank[c] * kRow);
          }
        if (lane == 0) {
          kr[0] = (uint32_t) nk;
          for (int b = 0; b <= g.nelt; b++) kr[1 + b] = (uint32_t) start[b];
        }
        wave_sync();
        descriptor_pass<K, NS>(g, cell, xi, pos, tab, nullptr, start, g.nelt, all, hb, Grow, 0, geo.g_bf16, true);
        return;
      }
    }
  }
  // phase 1: compaction
  const int nk = compact(g, cell, xi, (int) xi.w, nbr + (size_t) i * cap, nn[i], pos, kept, start);
  wave_sync();
  // the row's kept list with its slot starts, for the force kernel
  if (lane == 0) {
    kr[0] = (uint32_t) nk;
    for (int b = 0; b <= g.nelt; b++) kr[1 + b] = (uint32_t) start[b];
  }
  for (int e = lane; e < nk; e += 64) kr[kKeptHdr + e] = kept[e];
  if constexpr (!MP) {
    descriptor_pass<K, NS>(g, cell, xi, pos, tab, kept, start, g.nelt, rows, hb, Grow, 0, geo.g_bf16);
  } else {
    __shared__ int s_start[kMaxElts + 1];
    if (lane == 0)
      for (int b = 0; b <= g.nelt; b++) s_start[b] = start[b];
    wave_sync();
    for (int b0 = 0; b0 < g.nelt; b0 += NS)
      descriptor_pass<K, NS>(g, cell, xi, pos, tab, kept, s_start + b0, min(NS, g.nelt - b0), rows, hb, Grow, b0,
                             geo.g_bf16);
  }
}

// G row `row`; a padding row is cleared.  Returns its atom, or a negative number.
__device__ inline int descriptor_begin(const ModelGeo &g, const Geom &geo, int k, int row, const int *row2atom, float *G,
                                       float *&Grow)
{
  const int gw = g.nelt * k * kNM;
  // BF16 rows: gw 2-byte values per row (gw is a multiple of 4)
  Grow = geo.g_bf16 ? reinterpret_cast<float *>(reinterpret_cast<uint16_t *>(G) + (size_t) row * gw)
                    : G + (size_t) row * gw;
  const int i = row2atom[row];
  if (i < 0) {
    const int nw = geo.g_bf16 ? gw / 2 : gw;
    for (int e = threadIdx.x; e < nw; e += blockDim.x) Grow[e] = 0.0f;
  }
  return i;
}

// S = dE/dP of one slot from its P^T and dE/dG row (gslot[k][4]) -> sb
// [k][SS]: S_0 = g_0 (dropped below |G_0| = 1e-8, kernel.cu:754-759)
// + 2/3 g_2 P_0, S_d = 2 P_d (g_1 + 3/5 g_3 | g_2 | g_3) for degrees 1..3.
template <int K>
__device__ inline void slot_S(const f32x4v *p, const float4 *gv, int tsym, float *sb)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63, grp = lane >> 4;
#pragma unroll
  for (int t = 0; t < T::KT; t++) {
    const float4 v = gv[t];
    const float g2 = 2.0f * v.z, g3 = 2.0f * v.w;
    const float g1 = tsym ? 2.0f * v.y : fmaf(0.6f, g3, 2.0f * v.y);
    const float w0 = grp == 3 ? g3 : g2;                          // harmonic 4 grp (grp > 0)
    const float w1 = grp == 0 ? g1 : (grp == 1 ? g2 : g3);        // the other three
    const float g0 = fabsf(p[t][0]) < 1e-8f ? 0.0f : v.x;
    const float s0 = tsym ? g0 : fmaf(p[t][0], g2 * (1.0f / 3.0f), g0);
    const int k = 16 * t + (lane & 15);
    if (k < K)
      *reinterpret_cast<float4 *>(sb + k * T::SS + 4 * grp) =
          make_float4(grp == 0 ? s0 : p[t][0] * w0, p[t][1] * w1, p[t][2] * w1, p[t][3] * w1);
  }
}

// The S operands of one block for U (A[k][d], four MFMA steps of d = 4 g + s)
// and V (A[d][k], one step per filter of a lane group).
template <int K>
struct SOps {
  f32x4v u[Tiling<K>::CT];
  float v[Tiling<K>::NFB];
};

template <int K>
__device__ inline void load_S(const float *sb, int block, SOps<K> &o)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63, r = lane & 15, grp = lane >> 4;
  const float *s = sb + block * T::FBL * T::SS;
#pragma unroll
  for (int t = 0; t < T::CT; t++) {
    // the U row r of the accumulator is the filter nper(t) (r / 4) + r % 4 of
    // the tile (rows with r % 4 >= nper(t) repeat one and are not used)
    const int np = T::nper(t);
    const int f = 16 * t + (np == 4 ? r : 2 * (r >> 2) + (r & 1));
    o.u[t] = *reinterpret_cast<const f32x4v *>(s + f * T::SS + 4 * grp);
#pragma unroll
    for (int i = 0; i < np; i++) o.v[4 * t + i] = s[(16 * t + np * grp + i) * T::SS + r];
  }
}

// The chain rule of one block for a tile of neighbors (l % 16): f1 +=
// sum_k U_k dH_k over the lane group's filters, v += V
template <int K>
__device__ inline void chain_block(const SOps<K> &o, const f32x4v &y, const float *h, const float *dh, float &f1,
                                   f32x4v &v)
{
  using T = Tiling<K>;
#pragma unroll
  for (int t = 0; t < T::CT; t++) {
    f32x4v u = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++) u = __builtin_amdgcn_mfma_f32_16x16x4f32(o.u[t][s], y[s], u, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < T::nper(t); i++)
      v = __builtin_amdgcn_mfma_f32_16x16x4f32(o.v[4 * t + i], h[4 * t + i], v, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < T::nper(t); i++) f1 = fmaf(u[i], dh[4 * t + i], f1);
  }
}

// V and the lane group's f1 over the tile's harmonics and table offsets (the
// tile needs them no more; neighbors past the tile belong to other slots)
__device__ inline void put_V(float *rt, int live, float f1, const f32x4v &v)
{
  const int lane = threadIdx.x & 63, c = lane & 15, grp = lane >> 4;
  if (c < live) {
    *reinterpret_cast<f32x4v *>(rt + c * kRow + 4 * grp) = v;
    rt[c * kRow + kNY + grp] = f1;
  }
}

__device__ inline f32x4v get_Y(const float *rt, int live)
{
  const int lane = threadIdx.x & 63;
  return *reinterpret_cast<const f32x4v *>(rt + min(lane & 15, live - 1) * kRow + 4 * (lane >> 4));
}

// The force F of one neighbor (displacement d, atom j) from its V and f1 row;
// the row then holds F, j and, with vatom, -d (x) F for scatter(), and cf has own force
// and virial added.
struct ForceRow {
  double F[3];
  double v[6];
  int j;
};
static_assert(sizeof(ForceRow) <= kRow * sizeof(float) && kRow % 2 == 0, "a force row overlays a staged row");

__device__ inline void neighbor_force(const ModelGeo &g, const double d[3], int j, float *rowp, double scale,
                                      bool vatom, double *cf)
{
  const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
  const double ri = rsqrt_fp64(r2);
  const float x = (float) (d[0] * ri), y = (float) (d[1] * ri), z = (float) (d[2] * ri);
  float V[kNY];
  const float4 *r = reinterpret_cast<const float4 *>(rowp);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const float4 v = r[q];
    V[4 * q] = v.x;
    V[4 * q + 1] = v.y;
    V[4 * q + 2] = v.z;
    V[4 * q + 3] = v.w;
  }
  const float4 p = r[4];
  const float f1 = ((p.x + p.y) + (p.z + p.w)) * g.rdxf;
  float gx, gy, gz;
  harmonics_grad(x, y, z, V, gx, gy, gz);
  const float gu = gx * x + gy * y + gz * z;
  const float rinv = (float) ri;
  // dE_i/dd = F1 + F2; du_b/dd_a = (delta_ab - u_a u_b)/r
  const double F0 = (double) (f1 * x + (gx - gu * x) * rinv) * scale;
  const double F1 = (double) (f1 * y + (gy - gu * y) * rinv) * scale;
  const double F2 = (double) (f1 * z + (gz - gu * z) * rinv) * scale;
  const double v[6] = {-d[0] * F0, -d[1] * F1, -d[2] * F2, -d[0] * F1, -d[0] * F2, -d[1] * F2};
  ForceRow *o = reinterpret_cast<ForceRow *>(rowp);
  o->F[0] = F0;
  o->F[1] = F1;
  o->F[2] = F2;
  if (vatom) {
#pragma unroll
    for (int q = 0; q < 6; q++) o->v[q] = v[q];
  }
  o->j = j;
  cf[0] += F0;
  cf[1] += F1;
  cf[2] += F2;
#pragma unroll
  for (int q = 0; q < 6; q++) cf[3 + q] += v[q];
}

// f_j -= F (and the neighbor half of the per-atom virials) of the n neighbors
// in rows, FP64 atomics with adjacent lanes on adjacent components: they are
// executed at the memory side, one request per line of 64 bytes, and a
// neighbor's three components in three instructions were three requests
// (13.5 M requests and at least 640 us for the 24 M atomics of 128,000 atoms).
template <int W>
__device__ inline void scatter(const float *rows, int n, double *f, double *vatom)
{
  constexpr int lanes = 64 * W;
  const int lane = threadIdx.x & (lanes - 1);
  for (int t = lane; t < 3 * n; t += lanes) {
    const int c = t / 3, q = t - 3 * c;
    const ForceRow *o = reinterpret_cast<const ForceRow *>(rows + c * kRow);
    atomicAdd(&f[3 * (size_t) o->j + q], -o->F[q]);
  }
  if (vatom)
    for (int t = lane; t < 6 * n; t += lanes) {
      const int c = t / 6, q = t - 6 * c;
      const ForceRow *o = reinterpret_cast<const ForceRow *>(rows + c * kRow);
      atomicAdd(&vatom[6 * (size_t) o->j + q], 0.5 * o->v[q]);
    }
}

// facc += the lanes' own force and virial, in a fixed order.  Pairs of
// quantities share the exchanges between the halves and between the rows, so
// that four of them remain per register for the sums within a row of 16
// lanes.
__device__ inline void add_sums(const double *cf, double *facc)
{
  const int lane = threadIdx.x & 63;
  const double x0 = row_sum_d(swap16_add(swap32_add(cf[0], cf[1]), swap32_add(cf[2], cf[3])));
  const double x1 = row_sum_d(swap16_add(swap32_add(cf[4], cf[5]), swap32_add(cf[6], cf[7])));
  const double h8 = swap32_add(cf[8], cf[8]);
  const double x2 = row_sum_d(swap16_add(h8, h8));
  if ((lane & 15) == 0) {
    const int q = ((lane >> 4) & 1) * 2 + (lane >> 5);  // rows hold quantities 0, 2, 1, 3
    facc[q] += x0;
    facc[4 + q] += x1;
    if (lane == 0) facc[8] += x2;
  }
}

// dE/dG of one slot: filter l % 16 of every tile
template <int K>
__device__ inline void load_dEdG(const float *gslot, float4 *gv)
{
#pragma unroll
  for (int t = 0; t < Tiling<K>::KT; t++)
    gv[t] = *reinterpret_cast<const float4 *>(gslot + min(16 * t + (int) (threadIdx.x & 15), K - 1) * kNM);
}

// P += the staged neighbors rows[0..n) of one slot
template <int K>
__device__ inline void slot_moments(const float4 *tab, const float *rows, int n, float *hb, f32x4v *acc)
{
  using T = Tiling<K>;
  for (int r0 = 0; r0 < n; r0 += 16) {
    const int live = min(16, n - r0);
#pragma unroll
    for (int fb = 0; fb < T::NB; fb++) {
      TabTile<K> tt;
      load_tile<K>(tab, rows + r0 * kRow, live, fb, tt);
      put_H<K>(tt, hb);
      wave_sync();
      moments_tile<K, T::HS, 1>(rows + r0 * kRow, live, hb, acc + fb * T::CT);
      wave_sync();
    }
  }
}

// V and f1 of the staged neighbors rows[0..n) of one slot, over their rows.
// so: the slot's S operands where they fit registers, else read from sb.
template <int K>
__device__ inline void slot_chain(const float4 *tab, float *rows, int n, const float *sb,
                                  SOps<K> &so, float *hb)
{
  using T = Tiling<K>;
  for (int r0 = 0; r0 < n; r0 += 16) {
    const int live = min(16, n - r0);
    float *rt = rows + r0 * kRow;
    const f32x4v y = get_Y(rt, live);
    float f1 = 0.0f;
    f32x4v v = {0, 0, 0, 0};
#pragma unroll 1
    for (int fb = 0; fb < T::NB; fb++) {
      TabTile<K> tt;
      load_tile<K>(tab, rt, live, fb, tt);
      if constexpr (!T::kSRegs) load_S<K>(sb, fb, so);
      put_HD<K>(tt, hb);
      wave_sync();
      float h[T::NFB], dh[T::NFB];
      get_chain<K>(hb, h, dh);
      wave_sync();
      chain_block<K>(so, y, h, dh, f1, v);
    }
    put_V(rt, live, f1, v);
    wave_sync();
  }
}

// The forces of an atom whose kept list is longer than the staged window, by
// one wave.
template <int K, typename Start>
__device__ inline void force_long(const ModelGeo &g, const Box &cell, const double4 &xi, const double4 *pos,
                                  const float4 *tab, const uint32_t *kept, Start start, const float *grow,
                                  float *rows, float *hb, float *sb, double scale, double *f, double *vatom,
                                  double *facc)
{
  using T = Tiling<K>;
  const int lane = threadIdx.x & 63;
  // a longer list: slot by slot, P and then the chain rule in windows
  for (int b = 0; b < g.nelt; b++) {
    const int s0 = start(b), s1 = start(b + 1);
    if (s0 >= s1) continue;
    float4 gv[T::KT];
    load_dEdG<K>(grow + (size_t) b * K * kNM, gv);
    f32x4v acc[T::KT];
#pragma unroll
    for (int t = 0; t < T::KT; t++) acc[t] = f32x4v{0, 0, 0, 0};
    for (int w0 = s0; w0 < s1; w0 += T::WIN) {
      const int wn = min(T::WIN, s1 - w0);
      stage(g, cell, xi, pos, kept + w0, wn, rows);
      slot_moments<K>(tab, rows, wn, hb, acc);
    }
    slot_S<K>(acc, gv, g.tsym, sb);
    wave_sync();
    SOps<K> so;
    if constexpr (T::kSRegs) {
      load_S<K>(sb, 0, so);
      wave_sync();
    }
    for (int w0 = s0; w0 < s1; w0 += T::WIN) {
      const int wn = min(T::WIN, s1 - w0);
      if (s1 - s0 > T::WIN) stage(g, cell, xi, pos, kept + w0, wn, rows);
      slot_chain<K>(tab, rows, wn, sb, so, hb);
      double cf[9];
#pragma unroll
      for (int q = 0; q < 9; q++) cf[q] = 0.0;
      for (int c = lane; c < wn; c += 64) {
        const uint32_t e = kept[w0 + c];
        double d[3];
        displacement(xi, pos[e & kNbrJMask], e >> kNbrJBits, cell, d);
        neighbor_force(g, d, (int) (e & kNbrJMask), rows + c * kRow, scale, vatom, cf);
      }
      wave_sync();
      scatter<1>(rows, wn, f, vatom);
      add_sums(cf, facc);
      wave_sync();
    }
  }
}

}  // namespace

}  // namespace tmd
