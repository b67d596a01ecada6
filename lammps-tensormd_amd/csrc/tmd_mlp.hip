// Launch of the network kernels (tmd_mlp_kernels.h, one file per precision):
// LDS layout, tile rule, FP8 weight quantization.
#include "tmd_mlp_kernels.h"

#include <algorithm>

namespace tmd {

namespace {
__global__ void k_quant_fp8(const float *W, const float *swf, const float *swb, uint8_t *Af,
                            uint8_t *Ab, int K, int N, int nelt)
{
  const size_t per = (size_t) K * N;
  const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= per * nelt) return;
  const int el = (int) (i / per);
  const size_t rem = i - (size_t) el * per;
  const int k = (int) (rem / N), n = (int) (rem - (size_t) k * N);
  const float w = W[i];
  // forward operand: output n (tile n/16, lane row n%16), inner k (step
  // k/128, lane group (k%128)/32, byte k%32); backward: output k, inner n.
  // The B operands (quantize_rows, ld_x) place inner index k of a step at
  // the same lane group and byte, so the MFMA pairs equal k.
  const size_t f = (((size_t) (n / 16) * (K / 128) + k / 128) * 64 + ((k % 128) / 32) * 16 + n % 16) * 32 + k % 32;
  const size_t b = (((size_t) (k / 16) * (N / 128) + n / 128) * 64 + ((n % 128) / 32) * 16 + k % 16) * 32 + n % 32;
  Af[(size_t) el * per + f] =
      (uint8_t) (__builtin_amdgcn_cvt_pk_fp8_f32(w / swf[(size_t) el * N + n], 0.0f, 0, false) & 0xff);
  Ab[(size_t) el * per + b] =
      (uint8_t) (__builtin_amdgcn_cvt_pk_fp8_f32(w / swb[(size_t) el * K + k], 0.0f, 0, false) & 0xff);
}
}  // namespace

// every hidden width a multiple of 16 and every GEMM inner size a multiple of
// two fast-path steps (FP8: of one 128-wide step)
bool mlp_fast_ok(const MlpParams &mp, int mode)
{
  const int ks2 = mode == 0 ? 32 : (mode == 2 ? 128 : 64);
  for (int l = 0; l < mp.nl - 1; l++) {
    if (mp.sizes[l + 1] % 16 || mp.sizes[l] % 16) return false;
    if (mp.sizes[l] % ks2 || mp.sizes[l + 1] % ks2) return false;
  }
  return true;
}

hipError_t launch_quant_fp8(const float *W, const float *swf, const float *swb, uint8_t *Af,
                            uint8_t *Ab, int K, int N, int nelt, hipStream_t stream)
{
  size_t total = (size_t) K * N * nelt;
  if (total == 0) return hipSuccess;
  if (K % 32 || N % 32) return hipErrorInvalidValue;
  k_quant_fp8<<<(unsigned) ((total + 255) / 256), 256, 0, stream>>>(W, swf, swb, Af, Ab, K, N, nelt);
  return hipGetLastError();
}

// LDS layout for R rows: H_l and D_l per hidden layer (+ dE/dH for resnet).
size_t mlp_lds_bytes(const MlpParams &mp, int mode, int R, MlpParams *out)
{
  MlpParams m = mp;
  // FP32 activations in LDS for the FP32 and split-BF16 modes, BF16 for
  // the BF16 and FP8 modes
  const bool f32lds = mode == 0 || mode == 3;
  size_t esz = f32lds ? 4 : 2;
  size_t off = 0;
  int maxw = 0;
  bool anyres = false;
  for (int l = 0; l <= mp.nl - 1; l++) {
    int w = mp.sizes[l];
    m.ld[l] = R < 16 ? w + 16 : (f32lds ? w + 4 : w + 8);
  }
  for (int l = 0; l < mp.nl - 1; l++)
    if (mp.res[l]) anyres = true;
  // tanh without skips: D = 1 - h^2 is recomputed from H, so G_l overwrites H_l
  m.storeD = !(mp.act == 2 && !anyres);
  for (int l = 0; l < mp.nl - 1; l++) {
    int N = mp.sizes[l + 1];
    maxw = std::max(maxw, N);
    m.offH[l] = (int) off;
    off += (size_t) R * m.ld[l + 1];
    m.offD[l] = m.offH[l];
    if (m.storeD) {
      m.offD[l] = (int) off;
      off += (size_t) R * m.ld[l + 1];
    }
  }
  m.ldGH = R < 16 ? maxw + 16 : (f32lds ? maxw + 4 : maxw + 8);
  m.offGH = (int) off;
  if (anyres) off += (size_t) R * m.ldGH;
  // the fast kernel's staged descriptor rows: over the activations where the
  // first layer's outputs fit one pass of the waves, else behind them, or
  // not staged where that is too much
  m.stage_g = m.g_over = 0;
  m.offX = 0;
  m.ldx = m.ld[0];
  if (mode != 2 && mlp_fast_ok(mp, mode)) {
    const size_t xn = (size_t) R * m.ldx;
    if (mp.sizes[1] / 16 <= 4 * mlp_waves(mp, mode, R) && xn * esz <= 128 * 1024) {
      m.stage_g = m.g_over = 1;
      off = std::max(off, xn);
    } else if ((off + xn) * esz <= 80 * 1024) {
      m.stage_g = 1;
      m.offX = (int) off;
      off += xn;
    }
  }
  size_t bytes = (off * esz + 15) & ~(size_t) 15;
  m.offRS = (int) bytes;
  m.offQ = 0;
  m.ldq = 0;
  if (mode == 2) {
    bytes += 4 * (size_t) R * sizeof(float);  // scales, inverse scales, two buffers of recorded maxima
    // quantized B rows: the widest GEMM inner size, rows 16-byte aligned
    int maxk = 0;
    for (int l = 0; l < mp.nl; l++) maxk = std::max(maxk, mp.sizes[l]);
    m.ldq = maxk + 16;
    m.offQ = (int) ((bytes + 15) & ~(size_t) 15);
    bytes = (size_t) m.offQ + (size_t) R * m.ldq;
  }
  if (out) *out = m;
  return bytes;
}

bool mlp_bf16_rows(const MlpParams &mp, int mode)
{
  return mode == 1 && mlp_fast_ok(mp, 1) && mp.act == 2 && mlp_shape(mp) != 0;
}

namespace {
constexpr long kMlpLds = 160 * 1024;  // of a CU

// Rows per tile.  16 while 32-row tiles would not give every CU one (a tile
// is a serial chain of layers, and its length goes with its rows), or where
// only a tile of 16 has room for its descriptor rows in LDS (BF16
// 256-640-256-1, 16,000 rows: 74 us against 93 at 32); else 32.  64 in the
// BF16 mode once they give every CU two (half the weight reads), where two of
// them fit a CU: the compile-time shapes run four waves per SIMD at 64 rows
// (spilling 6 registers and 1; the other widths take 202), with at most 80 KB
// of LDS each.  384-256-256-128-1 has 83 KB: 128,000 rows take 218 us at 32
// rows and 257 at 64; 256-128-128-128-128-1 with skips 224 and 271.
// In the FP8 and split-BF16 modes, widths unknown at compile time: 16 or 32,
// whichever takes the chip fewer rounds of resident workgroups, 16 in a tie
// (FP8 1024-128-128-1, two and three workgroups per CU: 11,664 rows 42.9 at 16
// and 48.1 at 32 rows, 16,000 rows 66.0 and 55.4, 24,334 rows 84.5 and 97.2;
// split BF16 64-128-64-1: 16,384 rows 27.2 and 21.0).
// FP32 tiles of 4 and 8 rows while those give no CU a second one: a lone
// 16-row tile is bound by its CU's matrix cores, 0.11 us per 1,000 weights,
// so they pay where that is most of its time (16 K weights: 15.9 us at 16
// rows, 16.4 and 17.3 at 4 and 8; 82 K: 32.7, 29.5 and 32.4).  us, network
// alone, 384-256-128-64-1
// (139 K weights):     4 rows   8 rows  16 rows  32 rows  64 rows
//   FP32       128      18.3     23.5     32.5     52.0
//            1,024      22.1     24.3     32.6     52.4
//            2,000      30.9     29.0     35.0     53.8
//            3,456      53.6     38.4     38.5     55.6
//            8,192      95.6     68.7     56.7     58.8
//           16,000       184      127      105     93.5      103
//   BF16     2,000                        15.8     18.3     25.1
//            8,192                        25.0     25.5     32.1
//           16,000                        40.0     29.8     34.2
//           35,152                        73.2     66.5     65.1
//          128,000                         245      191      150
int tile_rows(const MlpParams &mp, int mode, int nrows, bool batch)
{
  if (mode == 0 && nrows <= 8 * kCUs && !batch) {
    long w = 0;
    for (int l = 0; l < mp.nl - 1; l++) w += (long) mp.sizes[l] * mp.sizes[l + 1];
    if (w >= 64 * 1024) return nrows <= 4 * kCUs ? 4 : 8;
  }
  if (mode >= 2 && !mlp_shape_kernel(mp, mode, 16)) {
    // rounds that the chip takes for all tiles, by its resident workgroups
    auto rounds = [&](int R) {
      const long lds = (long) mlp_lds_bytes(mp, mode, R, nullptr), fit = kMlpLds / lds;
      const long tiles = (nrows + R - 1) / R, held = kCUs * std::min(fit, mlp_waves(mp, mode, R) == 4 ? 3l : 1l);
      return held > 0 ? (tiles + held - 1) / held : tiles + 1;
    };
    return rounds(32) < rounds(16) ? 32 : 16;
  }
  if (nrows <= 32 * kCUs) return 16;
  MlpParams m16, m32;
  mlp_lds_bytes(mp, mode, 16, &m16);
  mlp_lds_bytes(mp, mode, 32, &m32);
  if (m16.stage_g && !m32.stage_g) return 16;
  if (mode == 1 && nrows >= 64 * 2 * kCUs && mlp_shape_kernel(mp, mode, 64) &&
      2 * (long) mlp_lds_bytes(mp, mode, 64, nullptr) <= kMlpLds)
    return 64;
  return 32;
}
}  // namespace

hipError_t launch_mlp(int mode, const RowLayout &rl, const MlpParams &mp, const float *G, double *E,
                      float *dEdG, hipStream_t s, int rtile, const BatchDims *dyn, int row_begin,
                      int row_end, bool g_bf16)
{
  if (g_bf16 && !mlp_bf16_rows(mp, mode)) return hipErrorInvalidValue;
  if (row_end < 0 || row_end > rl.nrows) row_end = rl.nrows;
  if (row_begin < 0 || row_begin > row_end) return hipErrorInvalidValue;
  if (row_end == row_begin) return hipSuccess;
  // rtile (16/32/64) overrides the rule; where its tile does not fit, the next
  // smaller of 32 and 16 rows
  int R = mlp_fast_ok(mp, mode) ? tile_rows(mp, mode, row_end - row_begin, dyn != nullptr) : 32;
  if (rtile == 16 || rtile == 32 || rtile == 64) R = rtile;
  for (;; R = R > 32 ? 32 : 16) {
    MlpParams m;
    const long lds = (long) mlp_lds_bytes(mp, mode, R, &m);
    // tiles of fewer than 16 rows read the descriptor rows from LDS only
    if (lds <= kMlpLds && (R >= 16 || m.stage_g)) {
      auto launch = mode == 0 ? launch_mlp_fp32 : (mode == 1 ? launch_mlp_bf16 : (mode == 2 ? launch_mlp_fp8 : launch_mlp_bf16x3));
      return launch(R, rl, m, G, E, dEdG, lds, s, dyn, row_begin, row_end, g_bf16);
    }
    if (R == 16) return hipErrorInvalidConfiguration;
  }
}

}  // namespace tmd
