// Internal interface between the host layer (tmd_api.cpp) and the gfx950
// kernels (tmd_device.hip).  All pointers are device pointers unless named
// h_*; every launcher enqueues on `stream` and returns hipError_t.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace tmd {

// Neighbor entries are one uint32: j in the low 23 bits, the image-shift code
// (s0+3)*49 + (s1+3)*7 + (s2+3), s in [-3, 3], in the top 9 bits.
constexpr int kNbrJBits = 23;
constexpr uint32_t kNbrJMask = (1u << kNbrJBits) - 1u;
constexpr int kMaxAtoms = (1 << kNbrJBits) - 1;
constexpr uint32_t kShiftCenter = 3u * 49u + 3u * 7u + 3u;
constexpr int kMaxElts = 8;
constexpr int kND = 20;  // monomials for max_moment 3
constexpr int kNM = 4;

// One periodic cell (a batch of structures has one per structure).  The
// neighbor-build fields are ignored by the descriptor/force kernels.
struct CellInfo {
  double h[9];    // rows a, b, c
  double inv[9];  // inverse (fractional = x * inv)
  int nb[3];      // bins per axis
  int reach[3];   // stencil half-width per axis
  int bin_base;   // first global bin of this cell
  int pad;
};

// Monomials of max_moment 3 in the order degree 0, 1, 2, 3 and, within a
// degree, x-power then y-power descending (tensormd.cpp:205-276): degree and
// multinomial multiplicity of monomial d.  T[m][d] = kMult[d] if kDeg[d] == m;
// a T-symmetric model adds T[2][0] = -1/3 and T[3][1..3] = -3/5.
constexpr int kDeg[kND] = {0, 1, 1, 1, 2, 2, 2, 2, 2, 2, 3, 3, 3, 3, 3, 3, 3, 3, 3, 3};
constexpr int kMult[kND] = {1, 1, 1, 1, 1, 2, 2, 1, 2, 1, 1, 3, 3, 3, 6, 3, 1, 3, 3, 1};

// Per-model constants passed by value to the descriptor/force kernels.
// slots[ei] packs the slot of neighbor element ej in bits 4ej..4ej+3
// (eltij of tensormd.cpp:165-176).
struct ModelGeo {
  int nelt;
  int k;
  int tab_n;
  int tsym;  // 1: T-symmetric descriptor
  int mm;    // max_moment as evaluated: 3 (0-2 are padded to 3), 4 or 5
  uint32_t slots[kMaxElts];
  double rc2;
  // grid step dx of the radial table: xdx finds the cell (the model's 1 / dx,
  // rounded to FP32 in a precision-32 model), rdx = 1 / dx scales offsets
  double xdx, rdx;
  float rdxf;
};

// Row layout of the MLP: rows are atoms grouped by element; each element
// group starts at a multiple of kRowTile.  row2atom[r] = -1 for padding.
constexpr int kRowTile = 64;
struct RowLayout {
  int nrows;                     // padded total
  int row_off[kMaxElts + 1];     // element e occupies [row_off[e], row_off[e+1])
};

// Sizes of one batch of structures, kept in device memory so that one
// captured graph (launched with grids sized for the capacities) serves
// every batch up to those capacities.  Kernels given a non-null BatchDims
// read their extents from it; workgroups beyond them exit at once.
struct BatchDims {
  int natoms;
  int nbins;
  int nstruct;
  int pad;
  RowLayout rl;
};

// The per-element MLP, all elements packed: layer l of element e starts at
// W*[l] + e * wstride[l].  Forward B operands: Wf32 = W [K][N] (fp32),
// Wtb = W^T [N][K] (bf16); backward: Wt32 = W^T [N][K] (fp32), Wb16 = W
// [K][N] (bf16).  The LDS fields are filled by the launcher.
constexpr int kMaxLayers = 8;
struct MlpParams {
  int nl;                        // layers including the width-1 output layer
  int sizes[kMaxLayers + 1];     // sizes[0] = descriptor width
  int act;
  int res[kMaxLayers];           // resnet skip of hidden layer l
  const float *Wf32[kMaxLayers];
  const float *Wt32[kMaxLayers];
  const uint16_t *Wtb[kMaxLayers];
  const uint16_t *Wb16[kMaxLayers];
  // fast path: the MFMA A operands of hidden layer l in the context's
  // precision (FP32, BF16, a BF16 hi + lo pair, or FP8 e4m3 divided by the
  // per-output-channel scale), stored in fragment order: tile t of 16 output channels, step s
  // of KS inner values, lane, then the lane's values, so that a wave loads
  // one fragment as one contiguous block.  Af: forward (outputs N, inner K),
  // Ab: backward (outputs K, inner N).  Element e at byte offset
  // e * wstride * (4, 2 or 1).
  const void *Af[kMaxLayers];
  const void *Ab[kMaxLayers];
  const float *swf[kMaxLayers];     // forward per-output-channel scales [N]
  const float *swb[kMaxLayers];     // backward per-output-channel scales [K]
  const float *b[kMaxLayers];    // hidden biases (or null)
  const float *wout;             // output layer weights [K_last]
  const float *bout;             // output bias (or null)
  long wstride[kMaxLayers];
  int bstride[kMaxLayers];
  // LDS layout (elements of the mode's type)
  int offH[kMaxLayers], offD[kMaxLayers], ld[kMaxLayers + 1];
  int offGH, ldGH;
  int offRS;   // FP8: per-row scale and inverse scale [2][R] (floats, byte offset)
  int offQ, ldq;  // FP8: the next GEMM's B operand rows, quantized [R][ldq] (bytes)
  int stage_g, g_over;  // descriptor rows staged in LDS; over the activations
  int offX, ldx;        // the staged rows [R][ldx]
  int storeD;  // D_l kept in LDS (otherwise recomputed from H_l: tanh)
};

// ---- neighbor build ---------------------------------------------------------
struct NbrBuild {
  int n;
  int cap;            // entries per atom
  double cut2;        // (rc + skin)^2
  double trig2;       // (skin/2)^2
  int nbins;          // total bins over all cells
  const CellInfo *cells;   // [ncells] (device)
  const int *atom_struct;  // [n] cell of each atom, or null (one cell)
  const BatchDims *dyn;    // device extents (n, nbins) when non-null
  int *bin_count;     // [nbins]
  int *bin_start;     // [nbins]
  int *bin_total;     // [1] atoms placed so far
  int *bin_atoms;     // [n]
  int *atom_bin;      // [n] flat bin
  int *atom_rank;     // [n] arrival rank in the bin
  int *atom_bc;       // [n][3] bin coordinates
  double4 *sorted;    // [n] positions in bin order, w = atom index
  double *x_build;    // [n][4]
  unsigned long long *ctl;  // [0] max d^2 bits, [1] force flag, [2] overflow, [3] build count, [5] batch error
};

// One neighbor-list update: a check (nbr_check, or launch_vv_first, which
// moves the atoms first), the rebuild kernels, which return at once when none
// is due, and at the end of the evaluation the reset of the control word
// (StepTail / launch_batch_finish).
hipError_t nbr_check(const NbrBuild &nb, const double4 *pos, hipStream_t stream);
// after_vv: launch_vv_first came before it on the same system
hipError_t nbr_rebuild(const NbrBuild &nb, double4 *pos, uint32_t *nbr, int *nn, hipStream_t stream,
                       bool after_vv = false);
// first half kick and drift, the displacement check, and f = 0; for a small
// system also the bins of a rebuild that is due
hipError_t launch_vv_first(const NbrBuild &nb, int n, double4 *pos, double *v, double *f, const double *dtfm,
                           double dt, hipStream_t stream);

// ---- descriptor / force -------------------------------------------------------
// Geometry of an evaluation: cells[atom_struct[i]] (atom_struct null: cells[0]).
struct Geom {
  const CellInfo *cells;
  const int *atom_struct;
  const BatchDims *dyn;  // rows beyond dyn->rl.nrows are skipped when non-null
  // the order in which the descriptor and force kernels take the rows: a
  // permutation of [0, nrows) (launch position p runs row order[p]); null:
  // row order.  Rows are element blocks, so atoms of one element run
  // together; the standalone system orders them by atom index instead,
  // which for spatially ordered atoms keeps neighboring atoms' work together
  const int *order = nullptr;
  // the descriptor kernel stores G as BF16 (round to nearest even, the BF16
  // MLP's own operand rounding) instead of FP32; max_moment <= 3 kernels only
  bool g_bf16 = false;
};
// The descriptor kernel's compaction of each row's list, reused by the force
// kernel of the same evaluation: kl[row][kKeptHdr + cap], kl[0] = nk,
// kl[1 + b] = first entry of slot b (b = 0..nelt), then the nk kept entries
// (within rc, sorted by slot).
constexpr int kKeptHdr = 16;
__host__ __device__ inline size_t kept_cache_words(int cap) { return (size_t) kKeptHdr + (size_t) cap; }

// Descriptor rows G[row] and the kept list of every row.
hipError_t launch_descriptor(const ModelGeo &g, const Geom &geo, const double4 *pos,
                             const uint32_t *nbr, const int *nn, int cap, const int *row2atom,
                             int nrows, const float4 *tab, float *G, uint32_t *kl,
                             hipStream_t stream, int row_begin = 0);

// Force/virial over the descriptor's kept lists: dEdG rows -> f (atomics,
// FP64, must be zeroed); per atom: eatom[i] = scale * E[row] and
// watom[i][6] = sum over the atom's pairs of -d (x) F (both written only for
// atoms that own a row); optional vatom (FP64 atomics; must be zeroed).
hipError_t launch_force(const ModelGeo &g, const Geom &geo, const double4 *pos, int cap,
                        const int *row2atom, int nrows, const float4 *tab, const uint32_t *kl,
                        const float *dEdG, const double *E, double scale, double *f, double *eatom,
                        double *watom, double *vatom, hipStream_t stream, int row_begin = 0);

// The same two kernels for max_moment 4 and 5 models (g.mm 4 or 5): 35 or 56
// monomials (tmd_desc_hm.hip); launch_descriptor/launch_force call them.
hipError_t launch_descriptor_hm(const ModelGeo &g, const Geom &geo, const double4 *pos,
                                const uint32_t *nbr, const int *nn, int cap, const int *row2atom,
                                int nrows, const float4 *tab, float *G, uint32_t *kl,
                                hipStream_t stream, int row_begin = 0);
hipError_t launch_force_hm(const ModelGeo &g, const Geom &geo, const double4 *pos, int cap,
                           const int *row2atom, int nrows, const float4 *tab, const uint32_t *kl,
                           const float *dEdG, const double *E, double scale, double *f,
                           double *eatom, double *watom, double *vatom, hipStream_t stream,
                           int row_begin = 0);

// Several waves per atom, for small systems (tmd_desc_wide.hip): the waves that
// the two kernels take for so many rows (1: the kernels of one wave), and
// the launches, which launch_descriptor/launch_force call.  Not for batches
// (Geom::dyn): their sums' order, and so a structure's last bits, must not
// depend on the batch's capacity.
bool desc_wide_ok(const ModelGeo &g, int rows);
int force_waves(const ModelGeo &g, int rows);
hipError_t launch_descriptor_wide(const ModelGeo &g, const Geom &geo, const double4 *pos, const uint32_t *nbr,
                                  const int *nn, int cap, const int *row2atom, int nrows, const float4 *tab, float *G,
                                  uint32_t *kl, hipStream_t stream, int row_begin);
hipError_t launch_force_wide(const ModelGeo &g, const Geom &geo, const double4 *pos, int cap, const int *row2atom,
                             int nrows, const float4 *tab, const uint32_t *kl, const float *dEdG, const double *E,
                             double scale, double *f, double *eatom, double *watom, double *vatom, hipStream_t stream,
                             int row_begin);

// ---- MLP ----------------------------------------------------------------------
// mode: 0 fp32, 1 bf16, 2 fp8 (e4m3 operands: weights with per-output-channel
// scales, activations and gradients with per-row scales; FP32 accumulation),
// 3 split bf16 (hi + lo operands, three BF16 products each).
// E[row] (FP64 output sum) and dEdG[row][width] (fp32).  rtile: rows per
// workgroup (16, 32 or 64; 0 = default).  The fast FP32 kernel takes 4 or 8 by
// default for few rows, which sums in another order than the larger tiles
// (those agree bit for bit): not with dyn, so that a structure's result does
// not depend on its batch's capacity.
// With dyn, rl gives the capacity (grid) and dyn->rl the live layout.
// Rows [row_begin, row_end) only (row_end < 0: to rl.nrows); both bounds
// are multiples of 64 (element blocks start on such rows).
// g_bf16: G holds BF16 rows (the descriptor kernel's Geom::g_bf16 output);
// only where mlp_bf16_rows() holds.
hipError_t launch_mlp(int mode, const RowLayout &rl, const MlpParams &mp, const float *G, double *E,
                      float *dEdG, hipStream_t stream, int rtile = 0,
                      const BatchDims *dyn = nullptr, int row_begin = 0, int row_end = -1,
                      bool g_bf16 = false);
// its precisions, at R rows per tile and with the LDS layout of mlp_lds_bytes
hipError_t launch_mlp_fp32(int R, const RowLayout &rl, const MlpParams &mp, const float *G, double *E, float *dEdG,
                           size_t lds, hipStream_t s, const BatchDims *dyn, int row_begin, int row_end, bool g_bf16);
hipError_t launch_mlp_bf16(int R, const RowLayout &rl, const MlpParams &mp, const float *G, double *E, float *dEdG,
                           size_t lds, hipStream_t s, const BatchDims *dyn, int row_begin, int row_end, bool g_bf16);
hipError_t launch_mlp_fp8(int R, const RowLayout &rl, const MlpParams &mp, const float *G, double *E, float *dEdG,
                          size_t lds, hipStream_t s, const BatchDims *dyn, int row_begin, int row_end, bool g_bf16);
hipError_t launch_mlp_bf16x3(int R, const RowLayout &rl, const MlpParams &mp, const float *G, double *E, float *dEdG,
                             size_t lds, hipStream_t s, const BatchDims *dyn, int row_begin, int row_end, bool g_bf16);
// the MLP launch takes BF16 descriptor rows: BF16 mode, tanh, a compile-time
// layer shape
bool mlp_bf16_rows(const MlpParams &mp, int mode);
size_t mlp_lds_bytes(const MlpParams &mp, int mode, int R, MlpParams *out);
// the fast (aligned) MLP kernel applies: required by the FP8 mode
bool mlp_fast_ok(const MlpParams &mp, int mode);
// FP8 A operands (MlpParams::Af/Ab layout) of one layer's weights for nelt
// elements: W [nelt][K][N] FP32, per-output-channel scales swf [nelt][N]
// (forward) and swb [nelt][K] (backward)
hipError_t launch_quant_fp8(const float *W, const float *swf, const float *swb, uint8_t *Af,
                            uint8_t *Ab, int K, int N, int nelt, hipStream_t stream);

// ---- TDNP: temperature-dependent models (src/ML-TENSORMD/tdnp.cpp) ------------------
// One network of every element: layer l of element e is W[l] + e K N
// ([K][N]), Wt[l] + e N K ([N][K]) and b[l] + e N (null without bias).
struct TdnpNet {
  int nl;
  int act;
  int sizes[kMaxLayers + 1];
  int res[kMaxLayers];
  const float *W[kMaxLayers];
  const float *Wt[kMaxLayers];
  const float *b[kMaxLayers];
};
// net[0] = H (descriptor -> ydim - 1, linear last layer), net[1] = U and
// net[2] = S (ydim -> 1); etemp: device scalar (eV), read at launch time.
struct TdnpParams {
  TdnpNet net[3];
  int ydim;
  int sommerfeld;
  const double *etemp;
};
// Per row: E[row] = u (FP64), sa[row] = {s, a} (FP64, a = u - T s), and
// dEdG[row] = dA/dG.  Padding rows get zeros.
hipError_t launch_tdnp(const RowLayout &rl, const TdnpParams &tp, const int *row2atom, const float *G,
                       double *E, double *sa, float *dEdG, hipStream_t stream,
                       const BatchDims *dyn = nullptr);

// ---- batches of structures (serving) ---------------------------------------------
// Capacities of one batch slot (grids of its captured graph).
struct BatchCaps {
  int atoms, rows, bins, structs;
  int nelt;  // model elements (valid element indices in pos.w)
};
// Device arrays of a batch slot.
struct BatchArrays {
  BatchDims *dyn;
  int *struct_off;    // [structs + 1]
  CellInfo *cells;    // [structs]
  int *atom_struct;   // [atoms]
  int *row2atom;      // [rows]
  double4 *pos;       // [atoms]
  double *f;                 // [atoms][3]
  const double *eatom;       // [atoms]
  const double *watom;       // [atoms][6]
  unsigned long long *ctl;   // neighbor control word
  int *bin_count, *bin_total;
};
// Dense host staging of a batch: BatchDims | struct_off[ns+1] | cells[ns] |
// atom_struct[n] | row2atom[nrows] | pos[n].  Byte offsets from the start:
// off[1] cells, off[2] atom_struct, off[3] row2atom, off[4] pos, off[5] and
// off[6] the total size (struct_off follows the header directly).
__host__ __device__ inline void batch_stage_offsets(int ns, int n, int nrows, size_t *off)
{
  auto up = [](size_t v) { return (v + 255) & ~(size_t) 255; };
  off[0] = 0;
  off[1] = up(sizeof(BatchDims) + 4 * (size_t) (ns + 1));
  off[2] = up(off[1] + sizeof(CellInfo) * (size_t) ns);
  off[3] = up(off[2] + 4 * (size_t) n);
  off[4] = up(off[3] + 4 * (size_t) nrows);
  off[5] = off[4] + sizeof(double4) * (size_t) n;
  off[6] = off[5];
}
// Dense host output of a batch: 8 header doubles (list overflow count,
// atoms, structures, error flag) | energy and virial[ns][7] | f[n][3] |
// eatom[n].
inline size_t batch_out_bytes(int ns, int n) { return 8 * (8 + 7 * (size_t) ns + 4 * (size_t) n); }
// Copy a staged batch (host memory, read by the kernels) into the slot's
// device arrays, clamping every count and index to the capacities; forces and
// bin counts of the batch are cleared.
hipError_t launch_batch_unpack(const void *stage, const BatchCaps &caps, const BatchArrays &a,
                               hipStream_t stream);
// Sum a finished batch's structures (fixed order), write its results to host
// memory `out` and reset the control word.
hipError_t launch_batch_finish(void *out, const BatchCaps &caps, const BatchArrays &a,
                               hipStream_t stream);

// ---- reductions / integration ---------------------------------------------------
hipError_t launch_zero(void *p, size_t bytes, hipStream_t stream);
// plain device-to-device copy (bandwidth calibration)
hipError_t launch_copy(const void *src, void *dst, size_t bytes, hipStream_t stream);
// What follows the force kernel of one evaluation: out[0] = sum_i eatom[i]
// and out[1..6] = sum_i watom[i][*] (fixed order; out holds 8 + 8 kSumParts
// doubles), the neighbor list's control word reset (ctl non-null), and, with
// v non-null, the second half kick of velocity Verlet and the kinetic energy
// sum(m v^2)/2 * mvv2e; with hist non-null the step's energies recorded at
// hist[2 n], n = (*counter)++ (safe to replay in a graph).
struct StepTail {
  const double *eatom, *watom;
  int n;
  double *out;
  unsigned long long *ctl;
  unsigned long long *ctl_host;  // with ctl: receives its 4 words (host memory)
  double trig2;
  const double4 *pos;
  double *v;
  const double *f, *dtfm, *mass;
  double *hist;
  unsigned long long *counter;
  int hist_cap;
};
constexpr int kSumParts = 240;
hipError_t launch_step_tail(const StepTail &t, hipStream_t stream);
// Host transfers of a system's state, through page-locked memory that the
// kernels read and write themselves.
// x [n][3] -> pos (elements kept) of atoms [first, first + n)
hipError_t launch_set_positions(int first, int n, const double *x, double4 *pos, unsigned long long *ctl,
                                hipStream_t stream);
// atoms [first, first + n) -> out: x [n][3], v [n][3], f [n][3], eatom [n],
// those asked for, one behind the other
struct StateOut {
  const double4 *pos;
  const double *v, *f, *eatom;
  double *out;
};
hipError_t launch_pack_state(int first, int n, const StateOut &s, hipStream_t stream);
// dst[0..n) = src[0..n), n <= 64
hipError_t launch_copy_small(const double *src, double *dst, int n, hipStream_t stream);
// pos, v and f to (save) or from snap [n](pos | v | f); counter = 0
hipError_t launch_snapshot(int n, bool save, double4 *pos, double *v, double *f, void *snap,
                           unsigned long long *counter, hipStream_t stream);
// *acc += sum of the kept-neighbor counts of the real rows (row2atom >= 0)
// in the kept-list cache kl (words per row)
hipError_t launch_sum_kept(const uint32_t *kl, size_t words, const int *row2atom, int nrows,
                           unsigned long long *acc, hipStream_t s);

}  // namespace tmd
