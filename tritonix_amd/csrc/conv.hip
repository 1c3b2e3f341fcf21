// C ABI of the conv2d forward path: argument checking, tile lookup, launch.
// Declarations and the reference interface they replace: include/tritonix_hip.h
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>

#include <new>
#include <unordered_map>

#include "../../include/tritonix_hip.h"
#include "conv_halo.h"
#include "conv_pack.h"
#include "conv_tile.h"
#include "registry.h"

using namespace tnx;

extern "C" const ConvGroup* tnx_conv_groups(int* ngroups);      // generated
extern "C" const KernelGroup* tnx_kernel_groups(int* ngroups);  // generated
extern "C" const GatherGroup* const* tnx_gather_groups(int* ngroups);  // generated
extern "C" const HaloEntry* const* tnx_halo_entries(int* n);    // generated

// The GEMM kernel's conv2d variant for this tile (three ring slots), or null.  Eight waves are preferred (and the
// only ones built): the loader's address arithmetic and the fix-up are vector instructions in the MFMA stream, and
// with two waves per SIMD one wave's arithmetic runs under the other's MFMAs (measured on 3x3 layers, batch 32,
// against four-wave builds: 256x128 524 -> 620 TFLOP/s at 56x56 / 256 channels, 128x128 248 -> 292 at 28x28 / 128
// and 351 -> 420 at 14x14 / 512).
static const KernelEntry* find_dma(int dtype, int bcout, int bpix, int bk) {
  int ng = 0;
  const KernelGroup* g = tnx_kernel_groups(&ng);
  const KernelEntry* four = nullptr;
  for (int i = 0; i < ng; ++i)
    for (int j = 0; j < g[i].count; ++j) {
      const KernelEntry& e = g[i].entries[j];
      if (e.dtype != dtype || e.bm != bcout || e.bn != bpix || e.bk != bk || e.stages != 3 || !e.conv) continue;
      if (e.nw == 8) return &e;
      if (e.nw == 4) four = &e;
    }
  return four;
}

static const ConvEntry* find_conv(int dtype, int bcout, int bpix, int bk) {
  int ng = 0;
  const ConvGroup* g = tnx_conv_groups(&ng);
  for (int i = 0; i < ng; ++i)
    for (int j = 0; j < g[i].count; ++j) {
      const ConvEntry& e = g[i].entries[j];
      if (e.dtype == dtype && e.block_cout == bcout && e.block_pix == bpix && e.block_k == bk) return &e;
    }
  return nullptr;
}

extern "C" void tnx_conv2d_output_size(const tnx_conv2d_args* a, int32_t* h_out, int32_t* w_out) {
  // floor division as Python's // does it (tritonix/ops/conv2d/forward.py:226-227)
  auto fdiv = [](int64_t x, int64_t d) { return x >= 0 ? x / d : -((-x + d - 1) / d); };
  int64_t h = 0, w = 0;
  if (a && a->stride_h > 0 && a->stride_w > 0) {
    h = fdiv((int64_t)a->h_in + 2 * (int64_t)a->pad_h - (int64_t)a->dil_h * (a->filter_h - 1) - 1, a->stride_h) + 1;
    w = fdiv((int64_t)a->w_in + 2 * (int64_t)a->pad_w - (int64_t)a->dil_w * (a->filter_w - 1) - 1, a->stride_w) + 1;
  }
  if (h_out) *h_out = (int32_t)h;
  if (w_out) *w_out = (int32_t)w;
}

// Measured on ResNet-style layers (3x3 / 1x1 / strided, 64-512 channels, batch 32): 64 pixels per tile is the
// fastest width everywhere -- the im2col loader's address arithmetic grows with the pixel width of the tile, the
// weight slab it shares the LDS with is reused from L2 -- and a 128-channel tile beats 64 whenever the layer has
// that many channels.
static void builtin_tile(const tnx_conv2d_args* a, int64_t pixels, int* bcout, int* bpix, int* bk) {
  (void)pixels;
  const int64_t gemm_k = (int64_t)a->c_in * a->filter_h * a->filter_w;
  *bcout = a->c_out > 64 ? 128 : 64;
  *bpix = 64;
  *bk = gemm_k > 32 ? 64 : 32;
}

// The image the direct-to-LDS kernel is given.  A 1x1 filter with unit strides and no padding reads whole planes
// in order, so the plane is handed over as one row of h*w pixels: the pixel index space then pads h*w, not every
// row, to a multiple of 8 (14x14: 200 columns per image instead of 224).  Only while h*w fits the kernel's 16-bit
// pixel coordinates.
struct DmaImage {
  int h_in, w_in, h_out, w_out, wp;
};
static DmaImage dma_image(const tnx_conv2d_args* a, int h_out, int w_out) {
  DmaImage g = {a->h_in, a->w_in, h_out, w_out, 0};
  if (a->filter_h == 1 && a->filter_w == 1 && a->stride_h == 1 && a->stride_w == 1 && a->pad_h == 0 && a->pad_w == 0 &&
      (int64_t)a->h_in * a->w_in <= 16384) {
    g.h_in = g.h_out = 1;
    g.w_in = g.w_out = a->h_in * a->w_in;
  }
  g.wp = (g.w_out + 7) / 8 * 8;
  return g;
}
static int64_t dma_cols(const tnx_conv2d_args* a, int h_out, int w_out) {
  const DmaImage g = dma_image(a, h_out, w_out);
  return (int64_t)a->batch * g.h_out * g.wp;
}

// Direct-to-LDS kernel: 256 channels x 128 pixels when that still leaves every CU two tiles, else 128 x 128.
// Measured on 3x3 layers (batch 32, eight-wave builds): 256x128 620 against 476 TFLOP/s for 128x128 at 56x56 / 256
// channels, 128x128 ahead of it at 28x28 / 128 channels (292 : 228) and 14x14 / 512 channels (420 : 337), and both
// well ahead of the register-staged kernel (392, 162, 165) down to a few dozen tiles.
static bool builtin_dma_tile(const tnx_conv2d_args* a, int h_out, int w_out, int* bcout, int* bpix, int* bk) {
  const int64_t cols = dma_cols(a, h_out, w_out);
  const int64_t t256 = ((cols + 127) / 128) * (((int64_t)a->c_out + 255) / 256);
  const int64_t t128 = ((cols + 127) / 128) * (((int64_t)a->c_out + 127) / 128);
  *bpix = 128;
  *bk = 64;
  if (a->c_out > 128 && t256 >= 512 && find_dma(a->dtype, 256, 128, 64)) {
    *bcout = 256;
    return true;
  }
  if (a->c_out > 64 && t128 >= 32 && find_dma(a->dtype, 128, 128, 64)) {
    *bcout = 128;
    return true;
  }
  return false;
}

// `rows` taps further along k = (c_in, fh, fw): rows = sc * (R*S) + sh * S + sw
static void tap_step(const tnx_conv2d_args* a, int rows, int hw_in, int* step_dw, int* step_dh, int* step_koff, int* lim_w,
                     int* lim_h, int* adj_w, int* adj_h) {
  const int rs = a->filter_h * a->filter_w;
  const int sc = rows / rs, sh = (rows % rs) / a->filter_w, sw = rows % a->filter_w;
  *step_dw = sw * a->dil_w;
  *step_dh = sh * a->dil_h;
  // (unsigned: for planes so large that `rows` channels further leaves the tensor the sum may wrap; such taps are
  // past the last k and never used)
  *step_koff = (int)((uint32_t)sc * (uint32_t)hw_in + (uint32_t)(*step_dh * a->w_in + *step_dw));
  *lim_w = a->filter_w * a->dil_w;
  *lim_h = a->filter_h * a->dil_h;
  *adj_w = a->dil_h * a->w_in - *lim_w;          // dw wraps: one filter row down
  *adj_h = hw_in - *lim_h * a->w_in;             // dh wraps: next input channel
}

// everything about the problem except the tile
static int check_problem(const tnx_conv2d_args* a, int32_t* h_out, int32_t* w_out) {
  if (!a) return TNX_E_INVALID;
  if (a->batch <= 0 || a->c_in <= 0 || a->h_in <= 0 || a->w_in <= 0 || a->c_out <= 0 || a->filter_h <= 0 ||
      a->filter_w <= 0 || a->stride_h <= 0 || a->stride_w <= 0 || a->pad_h < 0 || a->pad_w < 0 || a->dil_h <= 0 ||
      a->dil_w <= 0 || a->block_pixels < 0 || a->block_cout < 0 || a->block_k < 0 || a->group_pixels < 0)
    return TNX_E_INVALID;
  if (a->dtype == TNX_F32) return TNX_E_UNSUPPORTED;
  if (a->dtype != TNX_F16 && a->dtype != TNX_BF16) return TNX_E_INVALID;
  if (a->bias && a->bias_dtype != TNX_F16 && a->bias_dtype != TNX_BF16 && a->bias_dtype != TNX_F32) return TNX_E_INVALID;
  tnx_conv2d_output_size(a, h_out, w_out);
  if (*h_out <= 0 || *w_out <= 0) return TNX_E_INVALID;
  const int64_t lim = (1ll << 31) - 4096;
  const int64_t pixels = (int64_t)a->batch * *h_out * *w_out;
  const int64_t x_elems = (int64_t)a->batch * a->c_in * a->h_in * a->w_in;
  const int64_t w_elems = (int64_t)a->c_out * a->c_in * a->filter_h * a->filter_w;
  if (pixels >= lim || x_elems >= lim || w_elems >= lim) return TNX_E_UNSUPPORTED;
  if (a->h_in > 16384 || a->w_in > 16384 || a->pad_h > 16384 || a->pad_w > 16384 ||
      (int64_t)(a->filter_h - 1) * a->dil_h > 16384 || (int64_t)(a->filter_w - 1) * a->dil_w > 16384)
    return TNX_E_UNSUPPORTED;
  return TNX_OK;
}

// what the direct-to-LDS kernel needs of the problem (not of the tile)
static bool dma_problem_ok(const tnx_conv2d_args* a, int h_out, int w_out, bool inspect_ptrs) {
  const int64_t gemm_k = (int64_t)a->c_in * a->filter_h * a->filter_w;
  if (a->stride_w != 1 || gemm_k % 64 != 0) return false;
  if (dma_cols(a, h_out, w_out) >= (1ll << 31) - 4096) return false;
  if (inspect_ptrs && ((uintptr_t)a->weight & 15)) return false;
  // per-lane DMA offsets of the weight slab are 32-bit
  if (256 * gemm_k * 2 >= (1ll << 32)) return false;
  return true;
}

struct Resolved {
  const ConvEntry* reg;      // register-staged kernel, or
  const KernelEntry* dma;    // the GEMM kernel's conv2d variant, or
  bool gemm;                 // the plain GEMM kernel, one problem per image (1x1 filters, unit stride, no padding)
  int gemm_warps, gemm_stages;
  int bcout, bpix, bk;
  int h_out, w_out;
};

// A 1x1 filter with unit stride and no padding: out[n] = W[c_out, c_in] x X[n][c_in, h*w] + bias, image by image.
static bool gemm_problem_ok(const tnx_conv2d_args* a) {
  return a->filter_h == 1 && a->filter_w == 1 && a->stride_h == 1 && a->stride_w == 1 && a->pad_h == 0 && a->pad_w == 0;
}

// What a tile of that GEMM costs, in microseconds: `fixed` at its start and end, `slab` per K slab alone on its CU; of
// `per_cu` that share one, each one more adds `share` of the slabs' time; after whole rounds, a last one of few workgroups costs `last` of
// a whole one at least; `tail` for a last slab that is not whole; per 5 MB of output `store`, and `odd` more where rows of
// the output start off 16 bytes (narrow tiles then write more pieces of cache lines).  These loops are short: a CU that is done takes the
// next workgroup while others run, so a last round is counted at the mean number on a CU; counted at the most (last_round, further
// down) the choice measured 1.0210x the best tile on 1,500 layers, this way 1.0205x.
struct ImageCost {
  int bm, bn, nw, stages, per_cu;
  double fixed, slab, share, last, tail, store, odd;
};
static const ImageCost IMAGE_COST[] = {
    {128, 128, 8, 2, 2, 1.70, 0.408, 0.69, 0.97, 0.53, 0.69, 1.37},
    {128, 128, 8, 3, 1, 2.17, 0.323, 0.00, 1.00, 0.24, 0.97, 1.35},
    {64, 256, 8, 2, 2, 1.95, 0.611, 0.55, 0.77, 0.34, 0.44, 0.81},
    {128, 64, 8, 2, 3, 1.11, 0.271, 0.66, 0.95, 0.45, 0.97, 1.12},
    {128, 64, 8, 3, 2, 1.46, 0.200, 1.14, 0.90, 0.27, 1.06, 1.01},
    {64, 128, 8, 2, 3, 1.35, 0.398, 0.49, 0.83, 0.26, 0.74, 0.92},
    {64, 128, 8, 3, 2, 1.73, 0.301, 0.80, 0.72, 0.10, 0.75, 0.92},
    {64, 64, 4, 3, 3, 1.42, 0.227, 0.60, 0.76, 0.30, 0.67, 1.07},
    {32, 128, 4, 2, 4, 1.40, 0.346, 0.40, 0.84, 0.56, 0.40, 1.13},
    {32, 64, 4, 2, 6, 0.85, 0.206, 0.44, 0.66, 0.32, 1.05, 1.03},
    {32, 64, 4, 4, 3, 1.15, 0.142, 0.79, 0.63, 0.15, 0.89, 1.60}};

static double image_time(const ImageCost& c, const tnx_conv2d_args* a) {
  const int64_t hw = (int64_t)a->h_in * a->w_in, kt = (a->c_in + 63) / 64;
  const int64_t tiles = (((int64_t)a->c_out + c.bm - 1) / c.bm) * ((hw + c.bn - 1) / c.bn) * a->batch;
  const double k = (double)kt * c.slab * (a->c_in % 8 ? 1.23 : 1.0) * (hw % 8 ? 1.58 : 1.0);
  const double fixed = c.fixed + (a->c_in % 64 ? c.tail : 0.0);
  auto together = [&](double n) { return fixed + k * (1.0 + (n - 1.0) * c.share); };
  const int64_t slots = 256 * c.per_cu, full = tiles / slots, rem = tiles % slots;
  double t = (double)full * together(c.per_cu);
  if (rem && !full) t = together((double)((rem + 255) / 256));
  else if (rem) {
    const double n = (double)rem / 256.0;
    t += n < 1.0 ? together(1.0) * (c.last + (1.0 - c.last) * n) : together(n);
  }
  const double in = (double)a->batch * a->c_in * (double)hw * 2 / 5.0e6, out = (double)a->batch * a->c_out * (double)hw * (a->out_f32 ? 4 : 2) / 5.0e6;
  return 3.3 + 0.52 * in + t + (c.store + (hw % 8 ? c.odd : 0.0)) * out;
}

// Built-in tile for that GEMM.  128 x 128, narrowed to 64 channels or 64 pixels where the layer is that small or the grid would
// leave CUs idle, stays unless another one's modelled time is 5 % under its own: a least-squares fit to 11,720
// launches of 700 layers (1 to 128 images of 7x7 to 112x112, 3 to 2048 channels).  Measured on them it takes 0.927x the time
// of the first rule alone, 34 are slower by 3 % or more, 406 faster by 5 % or more: 16 images of 2034 channels, 14x14, 64 out:
// 23.7 -> 14.4 us (32x64 tiles, three on a CU); 128 of 23 channels, 33x33, 640 out: 136 -> 82 (64x256: longer runs of a row).
static bool builtin_gemm_tile(const tnx_conv2d_args* a, int* bcout, int* bpix, int* bk, int* nw, int* st) {
  const int64_t hw = (int64_t)a->h_in * a->w_in;
  int bm = a->c_out <= 64 ? 64 : 128, bn = hw <= 64 ? 64 : 128;
  auto tiles = [&](int m, int n) { return (((int64_t)a->c_out + m - 1) / m) * ((hw + n - 1) / n) * a->batch; };
  if (tiles(bm, bn) < 256 && bm > 64) bm = 64;
  if (tiles(bm, bn) < 256 && bn > 64) bn = 64;
  *bcout = bm; *bpix = bn; *bk = 64;
  if (!gemm_tile_for(a->dtype, bm, bn, 64, nw, st)) return false;
  // up to 16 channels out of one K slab in a round of tiles: every tile takes 4.5 to 5 us
  if (a->c_out <= 16 && a->c_in <= 64 && tiles(bm, bn) <= 256) return true;
  double best = 0.0;
  for (const ImageCost& c : IMAGE_COST)
    if (c.bm == bm && c.bn == bn && c.nw == *nw && c.stages == *st) best = 0.95 * image_time(c, a);
  for (const ImageCost& c : IMAGE_COST) {
    const double t = image_time(c, a);
    if (t < best) { best = t; *bcout = c.bm; *bpix = c.bn; *nw = c.nw; *st = c.stages; }
  }
  return true;
}

static void fill_gemm(const tnx_conv2d_args* a, const Resolved& r, tnx_gemm_args* g, GemmBatch* x) {
  const int64_t hw = (int64_t)a->h_in * a->w_in;
  *g = tnx_gemm_args{};
  g->a = a->weight; g->b = a->input; g->c = a->output;
  g->m = a->c_out; g->n = hw; g->k = a->c_in;
  g->stride_am = a->c_in; g->stride_ak = 1;
  g->stride_bk = hw; g->stride_bn = 1;
  g->stride_cm = hw; g->stride_cn = 1;
  g->in_dtype = a->dtype; g->out_dtype = a->out_f32 ? TNX_F32 : a->dtype;
  g->block_m = r.bcout; g->block_n = r.bpix; g->block_k = r.bk;
  g->group_m = 8; g->split_k = 1;
  g->num_stages = r.gemm_stages; g->num_warps = r.gemm_warps;
  g->epilogue = TNX_EPI_NONE;
  g->stream = a->stream;
  x->batch = a->batch;
  x->b_batch_bytes = (int64_t)a->c_in * hw * 2;
  x->c_batch_bytes = (int64_t)a->c_out * hw * (a->out_f32 ? 4 : 2);
  x->bias = a->bias;
  x->bias_dtype = a->bias_dtype;
}

static int resolve(const tnx_conv2d_args* a, Resolved* r, bool inspect_ptrs) {
  int32_t h_out = 0, w_out = 0;
  const int st = check_problem(a, &h_out, &w_out);
  if (st != TNX_OK) return st;
  if (a->loader < TNX_CONV_LOADER_AUTO || a->loader > TNX_CONV_LOADER_GEMM) return TNX_E_INVALID;
  const int64_t pixels = (int64_t)a->batch * h_out * w_out;
  const bool dma_ok = dma_problem_ok(a, h_out, w_out, inspect_ptrs);
  int bcout = a->block_cout, bpix = a->block_pixels, bk = a->block_k;
  const bool builtin = bcout == 0 && bpix == 0 && bk == 0;
  *r = Resolved{};
  r->h_out = h_out; r->w_out = w_out;
  if (a->loader == TNX_CONV_LOADER_GEMM && !gemm_problem_ok(a)) return TNX_E_UNSUPPORTED;
  // "auto" takes the GEMM route with the built-in tile (a caller's tile names a conv2d kernel) on every layer that is
  // such a GEMM: measured on the 1x1 layers of a ResNet-50 at batch 8, 32 and 128 it is level with or ahead of the
  // conv2d kernels on 34 of 36 (1.0x to 5.4x; 0.90x and 0.93x on 14x14 planes at batch 128, where it pads every image
  // to whole pixel tiles and the conv2d kernel packs the pixels of all images).
  const bool try_gemm = a->loader == TNX_CONV_LOADER_GEMM || (a->loader == TNX_CONV_LOADER_AUTO && builtin && gemm_problem_ok(a));
  if (try_gemm) {
    int nw = 0, st2 = 0;
    bool found = false;
    if (builtin) found = builtin_gemm_tile(a, &bcout, &bpix, &bk, &nw, &st2);
    else if (bcout > 0 && bpix > 0 && bk > 0) found = gemm_tile_for(a->dtype, bcout, bpix, bk, &nw, &st2);
    if (found) {
      r->gemm = true; r->gemm_warps = nw; r->gemm_stages = st2;
      r->bcout = bcout; r->bpix = bpix; r->bk = bk;
      tnx_gemm_args g;
      GemmBatch x;
      fill_gemm(a, *r, &g, &x);
      if (!inspect_ptrs) { g.a = nullptr; g.b = nullptr; g.c = nullptr; }
      const int sg = tnx_gemm_supported(&g);
      if (sg == TNX_OK && ((int64_t)((a->c_out + bcout - 1) / bcout) * (((int64_t)a->h_in * a->w_in + bpix - 1) / bpix) * a->batch < (1ll << 31)))
        return TNX_OK;
      if (a->loader == TNX_CONV_LOADER_GEMM) return sg == TNX_OK ? TNX_E_UNSUPPORTED : sg;
      r->gemm = false;
    } else if (a->loader == TNX_CONV_LOADER_GEMM) {
      return TNX_E_UNSUPPORTED;
    }
    bcout = a->block_cout; bpix = a->block_pixels; bk = a->block_k;
  }
  bool want_dma = a->loader == TNX_CONV_LOADER_DMA;
  if (builtin) {
    if (a->loader != TNX_CONV_LOADER_REGISTERS && dma_ok && builtin_dma_tile(a, h_out, w_out, &bcout, &bpix, &bk)) want_dma = true;
    else if (want_dma) return TNX_E_UNSUPPORTED;
    else builtin_tile(a, pixels, &bcout, &bpix, &bk);
  }
  if (bcout <= 0 || bpix <= 0 || bk <= 0) return TNX_E_INVALID;
  if (2ll * ((int64_t)bcout * bk + (int64_t)bk * bpix) * 2 > TNX_LDS_LIMIT_BYTES) return TNX_E_LDS;   // two slots: the smaller of the two kernels
  const ConvEntry* reg = find_conv(a->dtype, bcout, bpix, bk);
  const KernelEntry* dma = find_dma(a->dtype, bcout, bpix, bk);
  if (!builtin && a->loader == TNX_CONV_LOADER_AUTO) want_dma = dma && dma_ok;
  if (want_dma && !(dma && dma_ok)) {
    if (a->loader == TNX_CONV_LOADER_DMA) return TNX_E_UNSUPPORTED;
    want_dma = false;
  }
  if (!want_dma && !reg) return TNX_E_UNSUPPORTED;
  const int64_t cols = want_dma ? dma_cols(a, h_out, w_out) : pixels;
  if (((cols + bpix - 1) / bpix) * (((int64_t)a->c_out + bcout - 1) / bcout) >= (1ll << 31)) return TNX_E_UNSUPPORTED;
  r->reg = want_dma ? nullptr : reg;
  r->dma = want_dma ? dma : nullptr;
  r->bcout = bcout; r->bpix = bpix; r->bk = bk;
  r->h_out = h_out; r->w_out = w_out;
  return TNX_OK;
}

static void fill_registers(const tnx_conv2d_args* a, const Resolved& r, ConvParams* p, unsigned* grid) {
  const int h_out = r.h_out, w_out = r.w_out, bk = r.bk;
  const int64_t pixels = (int64_t)a->batch * h_out * w_out;
  const int64_t tiles_pix = (pixels + r.bpix - 1) / r.bpix, tiles_cout = ((int64_t)a->c_out + r.bcout - 1) / r.bcout;
  const int64_t gemm_k = (int64_t)a->c_in * a->filter_h * a->filter_w;
  const int64_t x_elems = (int64_t)a->batch * a->c_in * a->h_in * a->w_in;
  p->x = (const uint8_t*)a->input;
  p->w = (const uint8_t*)a->weight;
  p->bias = (const uint8_t*)a->bias;
  p->y = (uint8_t*)a->output;
  p->batch = a->batch; p->c_in = a->c_in; p->h_in = a->h_in; p->w_in = a->w_in;
  p->c_out = a->c_out; p->h_out = h_out; p->w_out = w_out; p->fh = a->filter_h; p->fw = a->filter_w;
  p->stride_h = a->stride_h; p->stride_w = a->stride_w; p->pad_h = a->pad_h; p->pad_w = a->pad_w;
  p->dil_h = a->dil_h; p->dil_w = a->dil_w;
  p->gemm_k = (int)gemm_k;
  p->pixels = (int)pixels;
  p->hw_in = a->h_in * a->w_in;
  p->hw_out = h_out * w_out;
  p->x_last_vec = (int)(x_elems - 8);
  p->x_bytes = (uint32_t)(x_elems * 2);
  p->w_bytes = (uint32_t)((int64_t)a->c_out * gemm_k * 2);
  p->div_hw_out = make_fastdiv((uint32_t)p->hw_out);
  p->div_w_out = make_fastdiv((uint32_t)w_out);
  p->div_rs = make_fastdiv((uint32_t)(a->filter_h * a->filter_w));
  p->div_s = make_fastdiv((uint32_t)a->filter_w);
  tap_step(a, bk, p->hw_in, &p->step_dw, &p->step_dh, &p->step_koff, &p->lim_w, &p->lim_h, &p->adj_w, &p->adj_h);
  p->tiles_cout = (int)tiles_cout;
  p->tiles_pix = (int)tiles_pix;
  p->group = a->group_pixels > 0 ? a->group_pixels : 8;
  p->bias_dtype = a->bias_dtype;
  p->w_vec_ok = gemm_k % 8 == 0 && ((uintptr_t)a->weight & 15) == 0;
  p->out_f32 = a->out_f32 != 0;
  p->y_vec_ok = p->hw_out % 4 == 0 && ((uintptr_t)a->output & (p->out_f32 ? 15 : 7)) == 0;
  p->flat = a->filter_h == 1 && a->filter_w == 1 && a->stride_h == 1 && a->stride_w == 1 && a->pad_h == 0 && a->pad_w == 0;
  *grid = (unsigned)(tiles_pix * tiles_cout);
}

// GemmParams of the GEMM kernel's conv2d variant: m = c_out, n = padded pixel index, k = c_in * R * S
static void fill_dma(const tnx_conv2d_args* a, const Resolved& r, GemmParams* p, unsigned* grid) {
  const DmaImage im = dma_image(a, r.h_out, r.w_out);
  const int h_out = im.h_out, w_out = im.w_out, wp = im.wp;
  const int64_t gemm_k = (int64_t)a->c_in * a->filter_h * a->filter_w;
  const int64_t n_total = (int64_t)a->batch * h_out * wp;
  memset(p, 0, sizeof *p);
  p->a = (const uint8_t*)a->weight;
  p->b = (const uint8_t*)a->input;
  p->c = (uint8_t*)a->output;
  p->m = a->c_out; p->n = n_total; p->k = gemm_k;
  p->sam = gemm_k; p->sak = 1;
  p->tiles_m = (int)(((int64_t)a->c_out + r.bcout - 1) / r.bcout);
  p->tiles_n = (int)((n_total + r.bpix - 1) / r.bpix);
  p->group_m = 8;            // with one or two channel tiles: the channel tiles of one pixel tile run side by side
  p->split_k = 1;
  p->ktiles_per_split = (int)(gemm_k / r.bk);
  p->out_dtype = a->out_f32 ? TNX_F32 : a->dtype;
  ConvGeom& g = p->cv;
  g.h_in = im.h_in; g.w_in = im.w_in; g.c_out = a->c_out; g.h_out = h_out; g.w_out = w_out; g.wp = wp;
  g.stride_h = a->stride_h; g.pad_h = a->pad_h; g.pad_w = a->pad_w;
  g.hw_in = a->h_in * a->w_in;
  g.chw_in = a->c_in * g.hw_in;
  g.n_total = (int)n_total;
  g.x_bytes = (uint32_t)((int64_t)a->batch * g.chw_in * 2);
  g.div_hwp = make_fastdiv((uint32_t)(h_out * wp));
  g.div_wp = make_fastdiv((uint32_t)wp);
  g.rs = a->filter_h * a->filter_w;
  g.fw = a->filter_w;
  g.div_rs = make_fastdiv((uint32_t)g.rs);
  g.div_s = make_fastdiv((uint32_t)g.fw);
  g.dil_h = a->dil_h; g.dil_w = a->dil_w;
  // the taps are tabulated slab by slab: one step is block_k rows
  tap_step(a, r.bk, g.hw_in, &g.step_dw, &g.step_dh, &g.step_koff, &g.lim_w, &g.lim_h, &g.adj_w, &g.adj_h);
  g.bias = (const uint8_t*)a->bias;
  g.bias_dtype = a->bias_dtype;
  *grid = (unsigned)((int64_t)p->tiles_m * p->tiles_n);
}

// ---------------------------------------------------------------------------
// packed route: one pass lays input and weight out (conv_pack.h), one GEMM launch over them.  Bound by the GEMM (MFMA and
// the start and end of its tiles) on wide layers, by the two launches on small ones.  Measured against the kernels that
// gather taps themselves, whole call, bf16/f16, 3x3: 256 channels of 56x56, batch 32: 155 -> 114 us (pass 18, GEMM 96:
// 1230 TFLOP/s); 128 channels of 56x56, stride 2: 42.8 -> 22.8; 512 of 7x7, batch 8: 137 -> 23; float32, 256 of 14x14: 242 -> 23.
// float32 with heads and tails in blocks of 32 channels instead of three terms (the GEMM reads a third less): 256 channels of
// 56x56, batch 32: 319 -> 301 us; 512 of 28x28: 285 -> 261; 128 of 56x56, stride 2: 53 -> 47; 512 of 7x7, batch 8: 39 -> 30.
// ---------------------------------------------------------------------------
// the window route (conv_halo.h), where it is taken instead: only the weight is laid out, and the workspace is the packed route's
struct HaloPlan {
  const HaloEntry* e;
  HaloGeom g;
  int lds, kt;                     // LDS of a workgroup; slabs of two k steps of a weight row
  int64_t w_bytes;
};

struct PackedPlan {
  const GatherEntry* e;
  HaloPlan halo;                   // halo.e null: not taken
  int split;                       // K slices per tile
  int h_out, w_out;
  int rows, cols, step_h, step_w;  // packed image; input rows / columns per packed row / column
  int terms, cp8, chunks, kt;      // bf16 terms per element; channel groups of 8 per term; k chunks; K slabs
  int hwp;
  int64_t n_total;
  int64_t slices_bytes, w_bytes, x_bytes;     // workspace: counters and K slices, weight, input
  int64_t total_bytes;
};

// What a packed tile costs, in microseconds: `fixed` at its start and end, `slab` per K slab alone on its CU; of `per_cu`
// that share one, each one more adds `share` of the slabs' time; `last` as in last_round.
struct GatherCost {
  int bm, bn, nw, stages, per_cu;
  double fixed, slab, share, last;
};
static const GatherCost GATHER_COST[] = {
    {256, 256, 8, 2, 1, 2.45, 1.163, 0.00, 0.96}, {256, 224, 8, 2, 1, 2.95, 1.058, 0.00, 0.91},
    {256, 192, 8, 2, 1, 2.51, 0.908, 0.00, 0.85}, {256, 128, 8, 3, 1, 2.15, 0.602, 0.00, 1.00},
    {128, 256, 8, 3, 1, 2.28, 0.620, 0.00, 0.92}, {128, 128, 8, 3, 1, 1.60, 0.350, 0.00, 1.00},
    {128, 128, 8, 2, 2, 0.79, 0.545, 0.31, 0.87}, {64, 256, 8, 3, 1, 1.80, 0.383, 0.00, 0.93},
    {64, 128, 8, 3, 2, 1.01, 0.258, 0.64, 0.78}, {64, 128, 8, 2, 2, 0.55, 0.459, 0.03, 0.95},
    {64, 128, 4, 3, 2, 1.17, 0.262, 0.55, 0.73}, {32, 256, 4, 2, 2, 0.89, 0.629, 0.02, 0.83},
    {64, 64, 4, 4, 2, 0.92, 0.141, 0.76, 0.90}, {64, 64, 4, 2, 4, 0.39, 0.386, 0.09, 0.87},
    {32, 128, 4, 3, 2, 0.89, 0.218, 0.45, 0.86}, {32, 128, 4, 2, 3, 0.43, 0.417, 0.10, 0.68},
    {32, 64, 4, 4, 2, 0.66, 0.119, 0.56, 1.00}};
// tile numbers of tnx_conv2d_packed_info / _forward: the first tiles of the table from 0, those of few channels or small rings from 32
static constexpr int FIRST_SMALL = 11, SMALL_FROM = 32;
static const GatherCost* gather_cost(const GatherEntry& e) {
  for (const GatherCost& c : GATHER_COST)
    if (c.bm == e.bm && c.bn == e.bn && c.nw == e.nw && c.stages == e.stages) return &c;
  return nullptr;
}

static constexpr double PAIR_SLAB = 1.3;
static constexpr double PASS_US = 9.0;     // the pass over the operands and the second launch, apart from the bytes

// Time of the last, partial round of `rem` workgroups: the CU that holds the most of them sets it.  After whole rounds, what it adds over
// a CU with one fewer counts from `last` (few such CUs) to whole (all of them).  (Counted at the mean number on a CU,
// 272 were 1.06 workgroups' time after a whole round and two workgroups' alone: 64 images of 256 channels, 28x28, 5x5, 62 out then
// took 784 tiles of 64x64 in place of 196 of 64x256, 74 us in place of 58.)
template <class F> static double last_round(F together, int64_t rem, bool after_whole, double last) {
  const int64_t most = (rem + 255) / 256;
  const double all = together((double)most);
  if (!after_whole) return all;
  const double fewer = most > 1 ? together((double)(most - 1)) : 0.0, part = (double)rem / 256.0 - (double)(most - 1);
  return fewer + (all - fewer) * (last + (1.0 - last) * part);
}

// Modelled microseconds of the GEMM over packed operands: `tiles` tiles of kt K slabs, cut `s` ways; `bytes` of input, as given
// and packed (what the caches cannot hold arrives up to a tenth slower).
static double gather_time(const GatherCost& c, int64_t tiles, int64_t kt, int s, bool pair, double bytes) {
  const double slow = 1.0 + 0.09 * (bytes < 3.0e8 ? bytes / 3.0e8 : 1.0);
  const double k = (double)((kt + s - 1) / s) * c.slab * (pair ? 1.05 : 1.0) * slow, area = c.bm * c.bn / 16384.0;
  const double fixed = c.fixed * (pair ? 1.98 : 1.0);
  auto together = [&](double n) { return fixed + k * (1.0 + (n - 1.0) * c.share); };
  const int64_t slots = 256 * c.per_cu, full = tiles * s / slots, rem = tiles * s % slots;
  double t = (double)full * together(c.per_cu);
  if (rem) t += last_round(together, rem, full > 0, c.last);
  if (s > 1) t += 1.6 + (0.13 + 0.42 * area) * s + 3.0 * (double)(tiles * s) * area / 256.0;
  return t;
}

// Modelled microseconds of the kernel a 16-bit layer has without scratch: rounds of workgroups x K slabs, constants fitted to
// 636 layers of 3x3 and 5x5 filters (two tiles of the register-staged kernel per CU cost it a third of its slab rate).
static double unpacked_time(const tnx_conv2d_args* a) {
  Resolved r;
  if (resolve(a, &r, false) != TNX_OK || r.gemm) return 1e300;
  const int64_t cols = r.dma ? dma_cols(a, r.h_out, r.w_out) : (int64_t)a->batch * r.h_out * r.w_out;
  const int64_t tiles = ((cols + r.bpix - 1) / r.bpix) * ((a->c_out + r.bcout - 1) / r.bcout);
  const double kt = (double)(((int64_t)a->c_in * a->filter_h * a->filter_w + r.bk - 1) / r.bk);
  if (r.dma) return 1.5 + (double)((tiles + 255) / 256) * (4.1 + (r.bcout > 128 ? 1.7 : 0.694) * kt);
  const double slots = r.bcout > 64 ? 320.0 : 800.0, rounds = tiles > slots ? tiles / slots : 1.0;
  return 4.0 + rounds * kt * (r.bcout > 64 ? 1.8 : tiles < 256 ? 1.15 + 0.4 * tiles / 256.0 : 1.55);
}

// Layers of few multiply-adds per output (packed_plan: `priced`): the packed route, its GEMM modelled at gemm_us, against the
// kernels that gather for themselves.  Both sides are least-squares fits to 782 such layers (10 % rms each); the choice costs
// 1.3 % against the better of the two in the mean, the line drawn at the multiply-adds alone cost 10 %.  Few channels out of
// a small plane stay with the one launch (3 channels of 17x17, 3x3, 45 out: 6.0 us, packed 9.6), many outputs do not (64 images of 3
// channels, 112x112, 3x3, 64 out: 115 us, packed 55; 128 of 36 channels, 56x56, 1x1 stride 2, 960 out: 200 and 79; float32,
// 64 of 19 channels, 17x17, 1x1, 1088 out: 49 and 36).  A call of two launches takes the host 11 to 12 us, one launch half of it: 16-bit
// layers under 12 us keep the one.  The float32 alternative is three launches on operands cut by two of them, 35 us and more
// for the host: below that it is never the faster call.
static bool few_taps_packed(const tnx_conv2d_args* a, const PackedPlan& p, double gemm_us, int h_out, int w_out) {
  const bool f32 = a->dtype == TNX_F32;
  const double es = f32 ? 4.0 : 2.0;
  const double out = (double)a->batch * a->c_out * h_out * w_out * es / 5.0e6;                 // in 5 MB: a microsecond of traffic
  const double in = (double)a->batch * a->c_in * a->h_in * a->w_in * es / 5.0e6;
  const double moved = (double)p.x_bytes / 5.0e6 + in / p.step_h, weight = (double)p.w_bytes / 5.0e6;
  const double packed = f32 ? 12.2 + 0.94 * gemm_us + 1.14 * out + 1.30 * moved + 1.04 * weight
                            : 8.7 + 0.92 * gemm_us + 1.12 * out + 1.62 * moved + 1.15 * weight;
  tnx_conv2d_args t = *a;
  if (f32) { t.dtype = TNX_BF16; t.c_in = 3 * a->c_in; }
  Resolved r;
  if (resolve(&t, &r, false) != TNX_OK) return true;
  if (f32 && packed <= 35.0) return true;
  if (r.gemm) return packed < 9.7 + 1.25 * out + 4.67 * in;
  const bool wide = r.bcout > 64;
  const int64_t tiles = (((int64_t)a->batch * h_out * w_out + r.bpix - 1) / r.bpix) * ((a->c_out + r.bcout - 1) / r.bcout);
  const double k32 = (double)(((int64_t)t.c_in * a->filter_h * a->filter_w + r.bk - 1) / r.bk * r.bk / 32);
  const double slots = 256.0 * (wide ? 1.53 : f32 ? 3.1 : 2.69), rounds = tiles > slots ? (double)tiles / slots : 1.0;
  const double alone = f32 ? (wide ? 9.9 : 7.8) + rounds * ((wide ? 0.0 : 1.8) + (wide ? 1.58 : 0.87) * k32) + 1.25 * out + 4.67 * in
                           : (wide ? 5.95 : 4.55) + rounds * ((wide ? 0.86 : 0.26) + (wide ? 0.80 : 0.84) * k32) + 3.06 * out + 0.57 * in;
  return packed < 0.95 * alone && alone >= 12.0;
}
static int64_t up256(int64_t v) { return (v + 255) / 256 * 256; }

// ---------------------------------------------------------------------------
// window route (conv_halo.h): 16-bit types, filters of at least two rows and columns, a column stride of at most 2
// ---------------------------------------------------------------------------
// Tile numbers of tnx_conv2d_packed_info / _forward: the window tiles from here on; `split` - 1 is then by how many groups of 8 pixels
// a tile is narrower than it could be.
static constexpr int HALO_FROM = 64;

// What a window tile costs, in microseconds: `fixed` at its start and end, `step` per k step (longer where short output rows make
// fragments straddle them), `event` per channel block in which all eight waves move rows; of up to `per_cu` that share a CU, as
// their LDS allows, each one more adds `share` of that; `last` as in last_round.
struct HaloCost {
  int bm, bn, ksp, slot, per_cu;
  double fixed, step, event, share, last;
};
static const HaloCost HALO_COST[] = {
    {256, 224, 2, 96, 1, 3.48, 0.430, 1.92, 0.00, 1.14}, {128, 192, 4, 96, 1, 2.78, 0.197, 1.08, 0.00, 1.00},
    {128, 128, 4, 96, 1, 2.37, 0.149, 0.97, 0.00, 1.02}, {64, 256, 4, 96, 1, 2.10, 0.148, 0.64, 0.00, 1.07},
    {64, 128, 4, 96, 2, 1.74, 0.100, 0.82, 0.65, 1.01}, {64, 64, 4, 96, 2, 1.71, 0.081, 1.08, 0.43, 0.95},
    {32, 256, 4, 96, 2, 1.99, 0.106, 0.71, 0.90, 1.05}, {32, 128, 4, 96, 2, 1.53, 0.080, 0.84, 0.47, 0.99},
    {128, 256, 2, 64, 1, 1.99, 0.301, 1.10, 0.00, 0.99}, {128, 128, 2, 64, 1, 2.00, 0.187, 1.13, 0.00, 0.99},
    {128, 128, 4, 64, 1, 2.30, 0.165, 0.91, 0.00, 0.98}, {64, 256, 4, 64, 1, 2.01, 0.169, 0.77, 0.00, 1.02},
    {64, 128, 4, 64, 2, 1.59, 0.110, 0.83, 0.62, 0.93}, {64, 64, 4, 64, 2, 1.64, 0.088, 1.01, 0.44, 0.87},
    {32, 256, 4, 64, 2, 1.65, 0.125, 0.81, 0.60, 0.92}, {32, 128, 4, 64, 2, 1.50, 0.091, 0.70, 0.44, 0.88}};

static int gcd(int a, int b) { while (b) { const int t = a % b; a = b; b = t; } return a; }

// What of the geometry is the layer's; false: not with any tile.
static bool halo_layer(const tnx_conv2d_args* a, int h_out, int w_out, HaloGeom* g) {
  if (a->filter_h < 2 || a->filter_w < 2 || a->stride_w > 2) return false;
  *g = HaloGeom{};
  g->c_in = a->c_in; g->h_in = a->h_in; g->w_in = a->w_in; g->plane = a->h_in * a->w_in;
  g->batch = a->batch; g->x_elems = (int)((int64_t)a->batch * a->c_in * g->plane);
  g->stride_h = a->stride_h; g->stride_w = a->stride_w; g->pad_h = a->pad_h; g->pad_w = a->pad_w;
  g->fh = a->filter_h; g->fw = a->filter_w; g->dil_h = a->dil_h; g->dil_w = a->dil_w; g->taps = a->filter_h * a->filter_w;
  g->blocks = (a->c_in + 31) / 32;
  const int64_t span = (int64_t)(a->filter_h - 1) * a->dil_h + 1, rows_img = (int64_t)(h_out - 1) * a->stride_h + span;
  const int64_t cols = (int64_t)(w_out - 1) * a->stride_w + (int64_t)(a->filter_w - 1) * a->dil_w + 1;
  // (a window of more than 4096 slots fits no LDS; k steps as far as their offsets do)
  if (g->x_elems < 8 || cols > 4096 || rows_img * a->batch >= (1ll << 31) || (int64_t)g->blocks * g->taps > 16384) return false;
  g->rows_img = (int)rows_img;
  g->cps = (int)((cols + a->stride_w - 1) / a->stride_w);
  g->rowslots = g->cps * a->stride_w;
  g->hw_out = h_out * w_out; g->hwp = (g->hw_out + 7) / 8 * 8; g->w_out = w_out;
  g->cpr = (a->w_in + 7) / 8;
  g->ksteps = g->blocks * g->taps;
  return true;
}

// Rows of the largest window of tiles of `width` pixels: from the first to the last pixel of a tile.  Inside an image the first pixel's
// column is a multiple of `step`; over c image ends each adds an image's rows and takes the pixels of one (hwp - hw_out of them lie in
// no row)
static int64_t halo_rows(const HaloGeom& g, int h_out, int width) {
  const int64_t span = (int64_t)(g.fh - 1) * g.dil_h + 1, rows_img = g.rows_img;
  const int w_out = g.w_out, common = gcd(width, g.hwp), step = gcd(common, w_out);
  int64_t most = (int64_t)((w_out - step + width - 1) / w_out) * g.stride_h;
  if (most > rows_img - span) most = rows_img - span;
  const int ends = (g.hwp - common + width - 1) / g.hwp;
  for (int c = 1; c <= ends; ++c) {
    const int left = width - 1 - c * g.hwp;             // pixels from the first one's place in its image to the last one's
    const int64_t down = (left >= 0 ? (left + w_out - 1) / w_out : -(-left / w_out)) + (g.hwp != g.hw_out ? 1 : 0);
    const int64_t d = c * rows_img + (down < h_out - 1 ? down : h_out - 1) * g.stride_h;
    if (d > most) most = d;
  }
  return most + span;
}

// The layer as tiles of `width` pixels, whose largest window has `rows` rows, see it, and the LDS of a workgroup; false: not with this tile.
static bool halo_tile(const HaloEntry& e, int width, int64_t rows, HaloGeom* g, int* lds) {
  // the next block's window has to wait for the block before the present one, and be there a period before its own first read
  if (g->ksteps <= e.ksp || (g->blocks > 1 && g->taps < 2 * e.ksp)) return false;
  const int64_t slots = rows * g->rowslots;
  if (slots > 4096 || rows * g->cpr > 128) return false;              // eight waves of 16 row pieces
  g->width = width;
  g->rows = (int)rows;
  g->buf_bytes = (int)(slots * e.slot);
  *lds = e.ring_bytes + 2 * g->buf_bytes + halo_table_bytes(e.ksp, (g->ksteps + e.ksp - 1) / e.ksp) + HALO_SPILL_BYTES;
  if (*lds < e.strip_bytes) *lds = e.strip_bytes;
  return *lds <= TNX_LDS_LIMIT_BYTES;
}

// Modelled microseconds of the route: a least-squares fit to 16,700 launches of 2,000 layers of 2x2 to 5x5 filters and 32 channels or
// more (7 % rms).
static double halo_time(const tnx_conv2d_args* a, const HaloCost& c, const HaloGeom& g, int64_t n_total, int lds) {
  const int64_t tiles = ((a->c_out + c.bm - 1) / c.bm) * ((n_total + g.width - 1) / g.width);
  const double weight = (double)a->c_out * a->c_in * g.taps * 2e-6 * (g.taps == 9 || g.taps == 25 ? 1.0 : 2.0);    // MB
  const double out = (double)a->batch * a->c_out * g.hw_out * 2 / 5.0e6, window = (double)g.rows * a->w_in * 64.0;
  const double body = g.ksteps * c.step * (1.0 + 1.80 / g.w_out) + g.blocks * c.event * ((g.rows * g.cpr + 15) / 16) / 8.0;
  const int fit = TNX_LDS_LIMIT_BYTES / lds, per_cu = fit < c.per_cu ? fit : c.per_cu;
  auto together = [&](double n) { return c.fixed + body * (1.0 + (n - 1.0) * c.share); };
  const int64_t slots = 256 * per_cu, full = tiles / slots, rem = tiles % slots;
  double t = (double)full * together(per_cu);
  if (rem) t += last_round(together, rem, full > 0, c.last);
  return 6.11 + 1.10 * weight + 0.87 * out + 0.061 * (double)tiles * window * g.blocks / 5.0e6 + t;
}

// Modelled microseconds of the packed route, its GEMM modelled at gemm_us (the same layers, 10 % rms): where a filter tap's channels are
// not whole slabs the GEMM reads the input tap after tap, from further away the larger it is, and rows that are not whole chunks
// cost both ends.
static double packed_time(const tnx_conv2d_args* a, double gemm_us, double x_bytes, double w_bytes, int h_out, int w_out) {
  const double in = (double)a->batch * a->c_in * a->h_in * a->w_in * 2 / 5.0e6, out = (double)a->batch * a->c_out * h_out * w_out * 2 / 5.0e6;
  const double far = x_bytes < 1.5e8 ? x_bytes / 5.0e7 : 3.0;
  return 8.38 + 1.01 * gemm_us * (a->c_in % 64 ? 1.0 + 0.142 * far : 1.0) + 1.63 * x_bytes / 5.0e6 + (a->w_in % 8 ? 0.52 * in : 0.0) +
         1.22 * w_bytes * 1e-6 + 0.74 * out * (w_out % 8 ? 1.69 : 1.0);
}

// tile >= 0: that tile of the type's table and that many K slices, whatever the rules below would choose
static bool make_packed_plan(const tnx_conv2d_args* a, PackedPlan* p, int tile, int split) {
  if (!a || a->loader != TNX_CONV_LOADER_AUTO || a->block_cout || a->block_pixels || a->block_k) return false;
  tnx_conv2d_args t = *a;
  const bool f32 = a->dtype == TNX_F32;
  if (f32) t.dtype = TNX_BF16;
  int32_t h_out = 0, w_out = 0;
  if (check_problem(&t, &h_out, &w_out) != TNX_OK) return false;
  if (f32 ? a->out_f32 == 0 : gemm_problem_ok(a)) return false;
  // The pass over the operands and a second launch do not always pay.  From 145 multiply-adds per output on (257 for a 1x1
  // filter, here with a stride, which reads every input element once either way) they did on all but 0.2 % of 654 layers; below
  // that the route is priced against the kernels that gather for themselves, further down.
  const int64_t macs = (int64_t)a->c_in * a->filter_h * a->filter_w;
  const bool priced = tile < 0 && macs <= (f32 ? 48 : a->filter_h * a->filter_w == 1 ? 256 : 144);
  if (tile >= 0 && (split < 1 || split > 16)) return false;
  *p = PackedPlan{};
  p->h_out = h_out; p->w_out = w_out;
  // a filter one row high reads only every stride_h-th input row: only those are packed (likewise for columns)
  p->step_h = a->filter_h == 1 ? a->stride_h : 1;
  p->step_w = a->filter_w == 1 ? a->stride_w : 1;
  const int sh = a->filter_h == 1 ? 1 : a->stride_h, sw = a->filter_w == 1 ? 1 : a->stride_w;
  p->rows = (h_out - 1) * sh + (a->filter_h - 1) * a->dil_h + 1;
  p->cols = (w_out - 1) * sw + (a->filter_w - 1) * a->dil_w + 1;
  p->cp8 = (a->c_in + 7) / 8;
  // float32: head and tail in blocks of 32 channels, one K slab each, or three terms of cp8 groups, 3/8 cp8 slabs.  A slab
  // of heads and tails takes three MFMA steps for two and measures about PAIR_SLAB of an ordinary one.  (25 to 32,
  // 49 to 64, 81 to 96, 105 to 128 and from 137 channels on.)
  const int blocks32 = (p->cp8 + 3) / 4;
  p->terms = !f32 ? 1 : PAIR_SLAB * blocks32 <= 0.375 * p->cp8 ? 2 : 3;
  if (p->terms == 2) p->cp8 = blocks32 * 4;
  const int64_t taps = (int64_t)a->filter_h * a->filter_w * p->terms;
  // the kernel's offset table has one entry per k chunk (it reads one slab past the end), or one per slab where a filter
  // tap's channels are whole slabs: a long k is padded to that
  if (p->cp8 * p->terms % 8 && ((taps * p->cp8 + 7) / 8 + 1) * 32 > GATHER_TABLE_BYTES) p->cp8 = (p->cp8 + 7) / 8 * 8;
  const int64_t chunks = taps * p->cp8, kt = (chunks + 7) / 8;
  if ((p->cp8 * p->terms % 8 ? (kt + 1) * 8 : kt + 1) * 4 > GATHER_TABLE_BYTES) return false;
  p->chunks = (int)chunks; p->kt = (int)kt;
  p->hwp = (h_out * w_out + 7) / 8 * 8;
  p->n_total = (int64_t)a->batch * p->hwp;
  p->x_bytes = (int64_t)a->batch * p->rows * p->cols * p->terms * p->cp8 * 16;
  p->w_bytes = (int64_t)a->c_out * kt * 128;
  const int64_t lim = (1ll << 31) - 4096;
  int nh = 0;
  const HaloEntry* const* he = tnx_halo_entries(&nh);
  HaloGeom layer;
  const bool windows = !f32 && (tile < 0 || tile >= HALO_FROM) && halo_layer(a, h_out, w_out, &layer);
  auto take_halo = [&](const HaloEntry* e, int width) {
    HaloPlan h = {e, layer};
    if (width < 8 || !halo_tile(*e, width, halo_rows(layer, h_out, width), &h.g, &h.lds)) return false;
    h.g.div_img = make_fastdiv((uint32_t)h.g.rows_img);
    h.g.div_hwp = make_fastdiv((uint32_t)h.g.hwp);
    h.g.div_w = make_fastdiv((uint32_t)w_out);
    h.g.div_cpr = make_fastdiv((uint32_t)h.g.cpr);
    h.g.div_taps = make_fastdiv((uint32_t)h.g.taps);
    h.g.div_fw = make_fastdiv((uint32_t)h.g.fw);
    h.kt = (h.g.ksteps + e->ksp - 1) / e->ksp * e->ksp / 2;           // whole periods
    h.w_bytes = (int64_t)a->c_out * h.kt * 128;
    if (p->n_total >= lim || h.w_bytes >= lim || ((a->c_out + e->bm - 1) / e->bm) * ((p->n_total + width - 1) / width) >= lim) return false;
    p->halo = h;
    return true;
  };
  if (tile >= HALO_FROM) {
    int left = tile - HALO_FROM;
    for (int i = 0; i < nh; ++i)
      if (windows && he[i]->dtype == a->dtype && left-- == 0 && take_halo(he[i], he[i]->bn - (split - 1) * 8)) {
        p->split = p->terms = 1;
        p->total_bytes = up256(p->halo.w_bytes);
        return true;
      }
    return false;
  }
  if (p->n_total >= lim || p->x_bytes >= lim || p->w_bytes >= lim || (int64_t)a->c_out * kt * 8 >= lim) return false;

  // Tile and K cut with the smallest modelled time (gather_time): constants and form are a least-squares fit to 112,000 measured
  // (layer, tile, cut) triples on 2,500 layers; on 1,600 others choosing by it costs 1.2 % against the best measured tile in the mean,
  // 7 % of them lose more than 5 %.
  // The tiles of 32 channels and those of two slots, several of which share a CU, win on layers of up to 64 channels and on
  // launches of many short tiles: 128 images of 64 channels, 28x28, 29 out: 28.5 -> 22 us, by 7 % on layers of up to 32
  // channels in the mean, by 3 % on the others.
  const double in_bytes = (double)p->x_bytes + (double)a->batch * a->c_in * a->h_in * a->w_in * (f32 ? 4 : 2) / p->step_h;
  double best = 1e300;
  int ng = 0, number = 0;
  const GatherGroup* const* g = tnx_gather_groups(&ng);
  for (int i = 0; i < ng; ++i)
    for (int j = 0; j < g[i]->count; ++j) {
      const GatherEntry& e = g[i]->entries[j];
      if (e.dtype != t.dtype) continue;
      if (tile >= 0) {
        if (number == FIRST_SMALL) number = SMALL_FROM;
        if (number++ == tile) { p->e = &e; p->split = split; }
        continue;
      }
      const GatherCost* cost = gather_cost(e);
      if (!cost) continue;
      const int64_t tiles = ((a->c_out + e.bm - 1) / e.bm) * ((p->n_total + e.bn - 1) / e.bn);
      for (int cut : {1, 2, 3, 4, 6, 8, 12, 16}) {
        if (cut > 1 && (kt / cut < 3 || tiles * cut > 800)) break;
        const int64_t per = (kt + cut - 1) / cut;
        const int s = (int)((kt + per - 1) / per);          // (no slice without a slab)
        const double c = gather_time(*cost, tiles, kt, s, p->terms == 2, in_bytes);
        if (c < best) { best = c; p->e = &e; p->split = s; }
      }
    }
  if (!p->e) return false;
  if (priced && !few_taps_packed(a, *p, best, h_out, w_out)) return false;
  // A wide padding (as a dilated filter has it) makes the packed image a multiple of the input, which the lines above do not
  // know.  From twice the input on the pass is priced, at the 5 TB/s it moves (what does not fit the memory-side cache costs the
  // GEMM twice its bytes more), against the kernel that needs none: 8 images of 2048 channels, 33x33 (packed 105x105), 256 out, 3x3:
  // 227 us packed, 209 not; 128 of 512, 7x7 (127x127), 64 out: 415 and 87; 1 of 2048, 33x33 (177x177), 256 out, 5x5: 52 and
  // 895.  On 636 layers of 1 to 6500 times the input, against the faster of the two: 0.4 % lost in the mean, 2.7 % without this
  // rule.  float32 stays: its alternative is an extra pass too.
  const double planes = (double)p->rows * p->cols / ((double)a->h_in * a->w_in);
  if (!f32 && tile < 0 && planes > 2.0) {
    const double bytes = (double)p->x_bytes + 2.0 * a->batch * (double)a->c_in * a->h_in * a->w_in;
    const double again = p->x_bytes > 200000000 ? 2.0 * ((double)p->x_bytes - 2.0e8) : 0.0;
    if (best + PASS_US + (bytes + again) / 5.0e6 > unpacked_time(&t)) return false;
  }
  // The window route where its modelled time is 10 % less (both models are off by 7 to 10 %), 17 % where w_out is no multiple of 8,
  // another 10 % for filters of two columns, and at least 0.88 of a channel block's 32 are channels: of the 2,000 layers 387 are
  // taken, which gain 25 % in the mean, 11 % over all layers of 40 us and more; 4 lose 3 % or more, the worst 9 %.  At 4 % without
  // the other lines 931 gain 16 % in the mean, 95 lose, the worst 28 % (128 images of 51 channels, 112x112, 5x5, 48 out: 359 us packed,
  // 387 as windows).  128 of 64, 28x28, 3x3, 64 out: 28.8 and 18.6; 32 of 256, 56x56, 256 out: 114 and 99; 32 of 128, 56x56, stride 2,
  // 128 out: 22.1 and 17.1; 32 of 512, 14x14, 512 out: 41.3 and 43.0.
  bool halo = false;
  if (windows && tile < 0 && a->c_in * 100 >= (a->c_in + 31) / 32 * 32 * 88) {
    const double margin = 0.9 * (w_out % 8 ? 0.92 : 1.0) * (a->filter_w == 2 ? 0.9 : 1.0);
    double best_halo = margin * packed_time(a, best, (double)p->x_bytes, (double)p->w_bytes, h_out, w_out);
    const HaloEntry* chosen = nullptr;
    int chosen_width = 0;
    int64_t rows_of[256 / 8 + 1] = {};           // by width / 8: most tiles share theirs
    for (int i = 0; i < nh; ++i) {
      const HaloEntry& e = *he[i];
      if (e.dtype != a->dtype) continue;
      const HaloCost* cost = nullptr;
      for (const HaloCost& c : HALO_COST)
        if (c.bm == e.bm && c.bn == e.bn && c.ksp == e.ksp && c.slot == e.slot) cost = &c;
      // tiles of whole output rows need fewer window rows (where images are whole tiles' worth of chunks, and not too much is given away)
      const int whole = e.bn / (w_out / gcd(w_out, 8) * 8) * (w_out / gcd(w_out, 8) * 8);
      const bool rows_too = whole < e.bn && whole >= 0.7 * e.bn && h_out * w_out % 8 == 0;
      for (int width : {e.bn, rows_too ? whole : 0}) {
        if (!cost || !width) continue;
        HaloGeom g = layer;
        int lds;
        if (!rows_of[width / 8]) rows_of[width / 8] = halo_rows(layer, h_out, width);
        if (!halo_tile(e, width, rows_of[width / 8], &g, &lds)) continue;
        const double t = halo_time(a, *cost, g, p->n_total, lds);
        if (t < best_halo) { best_halo = t; chosen = &e; chosen_width = width; }
      }
    }
    halo = chosen && take_halo(chosen, chosen_width);
  }
  const int64_t tiles = ((a->c_out + p->e->bm - 1) / p->e->bm) * ((p->n_total + p->e->bn - 1) / p->e->bn);
  if (tiles * p->split >= lim || (p->split > 1 && tiles > WS_MAX_TILES)) return false;
  p->slices_bytes = p->split > 1 ? WS_COUNTER_BYTES + (int64_t)p->split * tiles * p->e->bm * p->e->bn * 4 : 0;
  if (p->slices_bytes >= (1ll << 32)) return false;
  p->total_bytes = up256(p->slices_bytes) + up256(p->w_bytes) + up256(p->x_bytes);
  // (the workspace stays the packed route's: callers ask for it once, and what happens without room for it does not change)
  if (!halo || p->halo.w_bytes > p->total_bytes) p->halo.e = nullptr;
  return true;
}

// The library's own plans of the layers a thread has met, by their sizes: pricing one takes 2.1 us, finding it 0.1.  512 layers, more than
// a network has of different ones (at about 500 bytes each), and from the first again once they are full.
namespace {
struct LayerKey {
  int32_t v[22];
  bool operator==(const LayerKey& o) const { return memcmp(v, o.v, sizeof v) == 0; }
};
struct LayerHash {
  size_t operator()(const LayerKey& k) const {
    uint64_t h = 0x9e3779b97f4a7c15ull;
    for (int i = 0; i < 22; i += 2) {
      uint64_t w;
      memcpy(&w, k.v + i, 8);
      h = (h ^ w) * 0xff51afd7ed558ccdull;
      h ^= h >> 32;
    }
    return (size_t)h;
  }
};
struct KnownPlan {
  bool taken;
  PackedPlan plan;
};
constexpr size_t MOST_PLANS = 512;
}  // namespace

static bool packed_plan(const tnx_conv2d_args* a, PackedPlan* p, int tile = -1, int split = 1) {
  if (!a || tile >= 0) return make_packed_plan(a, p, tile, split);
  static thread_local std::unordered_map<LayerKey, KnownPlan, LayerHash> known;
  // (of a bias only whether its type is one that there is: the workspace is asked for without it)
  const bool odd_bias = a->bias && a->bias_dtype != TNX_F16 && a->bias_dtype != TNX_BF16 && a->bias_dtype != TNX_F32;
  const LayerKey key = {{a->batch, a->c_in, a->h_in, a->w_in, a->c_out, a->filter_h, a->filter_w, a->stride_h, a->stride_w, a->pad_h, a->pad_w,
                         a->dil_h, a->dil_w, a->dtype, a->out_f32 != 0, odd_bias, a->block_pixels, a->block_cout, a->block_k,
                         a->group_pixels, a->loader, 0}};
  const auto hit = known.find(key);
  if (hit != known.end()) {
    *p = hit->second.plan;
    return hit->second.taken;
  }
  *p = PackedPlan{};
  const bool taken = make_packed_plan(a, p, -1, 1);
  try {
    if (known.size() >= MOST_PLANS) known.clear();
    known.emplace(key, KnownPlan{taken, *p});
  } catch (const std::bad_alloc&) {              // no room to keep it: made again by the next call
  }
  return taken;
}

extern "C" size_t tnx_conv2d_workspace_bytes(const tnx_conv2d_args* a) {
  PackedPlan p;
  return packed_plan(a, &p) ? (size_t)p.total_bytes : 0;
}

static int halo_forward(const tnx_conv2d_args* a, const PackedPlan& pl) {
  const HaloEntry& e = *pl.halo.e;
  HaloGeom h = pl.halo.g;
  hipStream_t stream = (hipStream_t)a->stream;
  HaloWeight k;
  memset(&k, 0, sizeof k);
  k.w = (const uint8_t*)a->weight; k.out = (uint8_t*)a->workspace;
  k.c_in = a->c_in; k.c_out = a->c_out; k.groups = h.blocks * 4; k.chunks = pl.halo.kt * 8; k.taps = h.taps;
  k.div_groups = make_fastdiv((uint32_t)k.groups);
  const dim3 wgrid((unsigned)(((int64_t)k.c_out * k.groups + 63) / 64));
  if (k.taps == 9) hipLaunchKernelGGL(halo_weight_kernel<9>, wgrid, dim3(64), 0, stream, k);
  else if (k.taps == 25) hipLaunchKernelGGL(halo_weight_kernel<25>, wgrid, dim3(64), 0, stream, k);
  else hipLaunchKernelGGL(halo_weight_kernel<0>, wgrid, dim3(64), 0, stream, k);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) { note_hip_error((int)err); return TNX_E_HIP; }

  GemmParams p;
  memset(&p, 0, sizeof p);
  p.a = (const uint8_t*)a->workspace; p.c = (uint8_t*)a->output;
  p.m = a->c_out; p.n = pl.n_total; p.k = (int64_t)pl.halo.kt * 64;
  p.sam = p.k;
  p.tiles_m = (int)((a->c_out + e.bm - 1) / e.bm); p.tiles_n = (int)((pl.n_total + h.width - 1) / h.width);
  p.group_m = 8; p.split_k = 1;
  p.out_dtype = a->out_f32 ? TNX_F32 : a->dtype;
  // the output side is conv2d's epilogue on planes of one row of hwp pixels
  ConvGeom& c = p.cv;
  c.c_out = a->c_out; c.h_out = 1; c.w_out = h.hw_out; c.wp = pl.hwp;
  c.n_total = (int)pl.n_total;
  c.div_hwp = c.div_wp = make_fastdiv((uint32_t)pl.hwp);
  c.bias = (const uint8_t*)a->bias;
  c.bias_dtype = a->bias_dtype;
  h.x = (const uint8_t*)a->input;
  err = e.launch(p, h, (unsigned)((int64_t)p.tiles_m * p.tiles_n), pl.halo.lds, stream);
  if (err != hipSuccess) { note_hip_error((int)err); return TNX_E_HIP; }
  return TNX_OK;
}

static int packed_forward(const tnx_conv2d_args* a, const PackedPlan& pl) {
  if (pl.halo.e) return halo_forward(a, pl);
  uint8_t* ws = (uint8_t*)a->workspace;
  uint8_t* wp = ws + up256(pl.slices_bytes);
  uint8_t* xp = wp + up256(pl.w_bytes);
  const int cpt = pl.cp8 * pl.terms;
  const bool f32 = a->dtype == TNX_F32;
  const GatherEntry& e = *pl.e;
  const int64_t tiles_m = (a->c_out + e.bm - 1) / e.bm, tiles_n = (pl.n_total + e.bn - 1) / e.bn;

  PackParams k;
  memset(&k, 0, sizeof k);
  k.x = (const uint8_t*)a->input; k.w = (const uint8_t*)a->weight; k.xp = xp; k.wp = wp;
  if (pl.split > 1) { k.counters = (int*)ws; k.ncounters = (int)(tiles_m * tiles_n); }
  k.c_in = a->c_in; k.h_in = a->h_in; k.w_in = a->w_in; k.taps = a->filter_h * a->filter_w;
  k.rows = pl.rows; k.cols = pl.cols; k.step_h = pl.step_h; k.step_w = pl.step_w;
  k.pad_h = a->pad_h; k.pad_w = a->pad_w;
  k.cp8 = pl.cp8; k.chunks = pl.chunks; k.chunks_pad = pl.kt * 8;
  // columns that can hold input: the chunks cover those, `lead` padding columns before them
  k.lead = pl.step_w == 1 && a->pad_w < pl.cols ? a->pad_w : 0;
  const int inside = pl.step_w == 1 && a->pad_w < pl.cols ? (a->w_in < pl.cols - k.lead ? a->w_in : pl.cols - k.lead) : pl.cols;
  k.wchunks = (inside + 7) / 8;
  k.whole = cpt % 8 == 0;
  k.div_taps = make_fastdiv((uint32_t)(a->filter_h * a->filter_w));
  k.cgb = (pl.cp8 + 7) / 8;
  const int per_wave = 64 >> pack_cg_bits(pl.cp8);
  const int64_t x_items = (int64_t)a->batch * pl.rows * k.wchunks, waves = (x_items + per_wave - 1) / per_wave * k.cgb;
  const int64_t w_items = (int64_t)a->c_out * k.chunks_pad;
  if (x_items >= (1ll << 31) || waves >= (1ll << 31)) return TNX_E_UNSUPPORTED;
  k.x_items = (int)x_items;
  k.w_items = (int)w_items;
  k.x_elems = (int)((int64_t)a->batch * a->c_in * a->h_in * a->w_in);
  const int64_t w_threads = w_items > k.ncounters ? w_items : k.ncounters;
  k.w_blocks = (unsigned)((w_threads + 255) / 256);
  k.div_cgb = make_fastdiv((uint32_t)k.cgb);
  k.div_row = make_fastdiv((uint32_t)pl.rows);
  k.div_wchunks = make_fastdiv((uint32_t)k.wchunks);
  k.div_cpt = make_fastdiv((uint32_t)cpt);
  k.div_cp8 = make_fastdiv((uint32_t)pl.cp8);
  k.div_chunks = make_fastdiv((uint32_t)k.chunks_pad);
  const unsigned blocks = k.w_blocks + (unsigned)((waves + 3) / 4);
  hipStream_t stream = (hipStream_t)a->stream;
  const bool unit = pl.step_w == 1;
  void (*pack)(PackParams) = !f32 ? (unit ? conv_pack_kernel<uint16_t, 1, true> : conv_pack_kernel<uint16_t, 1, false>)
                             : pl.terms == 2 ? (unit ? conv_pack_kernel<float, 2, true> : conv_pack_kernel<float, 2, false>)
                                             : (unit ? conv_pack_kernel<float, 3, true> : conv_pack_kernel<float, 3, false>);
  hipLaunchKernelGGL(pack, dim3(blocks), dim3(256), 0, stream, k);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) { note_hip_error((int)err); return TNX_E_HIP; }

  GemmParams p;
  memset(&p, 0, sizeof p);
  p.a = wp; p.b = xp; p.c = (uint8_t*)a->output; p.ws = ws;
  p.m = a->c_out; p.n = pl.n_total; p.k = (int64_t)pl.kt * 64;
  p.sam = p.k; p.sak = 1; p.sbk = 1; p.sbn = 0;
  p.tiles_m = (int)tiles_m; p.tiles_n = (int)tiles_n;
  p.group_m = 8;
  p.split_k = pl.split;
  p.ktiles_per_split = (pl.kt + pl.split - 1) / pl.split;
  p.out_dtype = f32 || a->out_f32 ? TNX_F32 : a->dtype;
  const int hw_out = pl.h_out * pl.w_out;
  // the output side is conv2d's epilogue on planes of one row of hwp pixels
  ConvGeom& g = p.cv;
  g.c_out = a->c_out; g.h_out = 1; g.w_out = hw_out; g.wp = pl.hwp;
  g.n_total = (int)pl.n_total;
  g.div_hwp = g.div_wp = make_fastdiv((uint32_t)pl.hwp);
  g.bias = (const uint8_t*)a->bias;
  g.bias_dtype = a->bias_dtype;
  PackGeom& q = p.pk;
  q.hw_out = hw_out; q.hwp = pl.hwp; q.w_out = pl.w_out;
  q.div_hwp = g.div_hwp; q.div_w = make_fastdiv((uint32_t)pl.w_out);
  const uint32_t px = (uint32_t)cpt * 16u;             // bytes of one packed pixel
  q.img_bytes = (uint32_t)pl.rows * (uint32_t)pl.cols * px;
  q.row_bytes = (uint32_t)(a->filter_h == 1 ? 1 : a->stride_h) * (uint32_t)pl.cols * px;
  q.col_bytes = (uint32_t)(a->filter_w == 1 ? 1 : a->stride_w) * px;
  q.chunks = pl.chunks; q.cpt = cpt; q.fw = a->filter_w; q.taps = a->filter_h * a->filter_w;
  q.div_taps = k.div_taps;
  q.div_cpt = k.div_cpt; q.div_fw = make_fastdiv((uint32_t)a->filter_w);
  q.tap_row_bytes = (uint32_t)a->dil_h * (uint32_t)pl.cols * px;
  q.tap_col_bytes = (uint32_t)a->dil_w * px;
  q.x_bytes = (uint32_t)pl.x_bytes;
  err = (pl.terms == 2 ? e.pair : e.launch)(p, (unsigned)(tiles_m * tiles_n * pl.split), stream);
  if (err != hipSuccess) { note_hip_error((int)err); return TNX_E_HIP; }
  return TNX_OK;
}

extern "C" size_t tnx_conv2d_packed_info(const tnx_conv2d_args* a, int tile, int split, int32_t* info) {
  PackedPlan p;
  if (!packed_plan(a, &p, tile, split)) return 0;
  if (info) {
    const HaloEntry* w = tile >= 0 ? p.halo.e : nullptr;
    const int32_t v[6] = {w ? w->bm : p.e->bm, w ? w->bn : p.e->bn, w ? 8 : p.e->nw, w ? w->ring : p.e->stages, w ? p.halo.g.rows : p.split, w ? p.halo.lds : p.terms};
    memcpy(info, v, sizeof v);
  }
  return (size_t)p.total_bytes;
}

// the checks of a launch that has a plan and a workspace
static int packed_launch(const tnx_conv2d_args* a, const PackedPlan& pl) {
  if (!a->workspace || a->workspace_bytes < (size_t)pl.total_bytes || ((uintptr_t)a->workspace & 255)) return TNX_E_WORKSPACE;
  const unsigned in_align = a->dtype == TNX_F32 ? 3 : 1, out_align = a->out_f32 ? 3 : 1;
  if (!a->input || !a->weight || !a->output || ((uintptr_t)a->input & in_align) || ((uintptr_t)a->weight & in_align) ||
      ((uintptr_t)a->output & out_align) || (a->bias && ((uintptr_t)a->bias & (a->bias_dtype == TNX_F32 ? 3 : 1))))
    return TNX_E_INVALID;
  return packed_forward(a, pl);
}

extern "C" int tnx_conv2d_packed_forward(const tnx_conv2d_args* a, int tile, int split) {
  PackedPlan pl;
  if (!packed_plan(a, &pl, tile, split)) return TNX_E_UNSUPPORTED;
  if (tile < 0) pl.halo.e = nullptr;           // this route's tile, whichever the layer takes
  return packed_launch(a, pl);
}

extern "C" int tnx_conv2d_route(const tnx_conv2d_args* a, int32_t info[3]) {
  PackedPlan pl;
  Resolved r;
  int route = 0, tile[3] = {0, 0, 1};
  if (a && a->workspace && packed_plan(a, &pl)) {
    const HaloEntry* w = pl.halo.e;
    route = w ? TNX_CONV_ROUTE_WINDOW : TNX_CONV_ROUTE_PACKED;
    tile[0] = w ? w->bm : pl.e->bm;
    tile[1] = w ? pl.halo.g.width : pl.e->bn;
    tile[2] = w ? 1 : pl.split;
  } else if (resolve(a, &r, true) == TNX_OK) {
    route = r.gemm ? TNX_CONV_ROUTE_GEMM : r.dma ? TNX_CONV_ROUTE_DMA : TNX_CONV_ROUTE_REGISTERS;
    tile[0] = r.bcout;
    tile[1] = r.bpix;
  }
  if (info && route) memcpy(info, tile, sizeof tile);
  return route;
}

extern "C" int tnx_conv2d_supported(const tnx_conv2d_args* a) {
  Resolved r;
  return resolve(a, &r, false);
}

extern "C" int tnx_conv2d_default_config(tnx_conv2d_args* a) {
  if (!a) return TNX_E_INVALID;
  tnx_conv2d_args tmp = *a;
  tmp.block_cout = tmp.block_pixels = tmp.block_k = 0;
  Resolved r;
  const int st = resolve(&tmp, &r, a->weight != nullptr);     // a weight pointer, when given, is checked for alignment
  if (st != TNX_OK) return st;
  a->block_cout = r.bcout;
  a->block_pixels = r.bpix;
  a->block_k = r.bk;
  a->group_pixels = 8;
  a->loader = r.gemm ? TNX_CONV_LOADER_GEMM : r.dma ? TNX_CONV_LOADER_DMA : TNX_CONV_LOADER_REGISTERS;
  return TNX_OK;
}

extern "C" int tnx_conv2d_forward(const tnx_conv2d_args* a) {
  if (a && a->workspace) {
    PackedPlan pl;
    if (packed_plan(a, &pl)) return packed_launch(a, pl);
  }
  Resolved r;
  const int st = resolve(a, &r, true);
  if (st != TNX_OK) return st;
  if (!a->input || !a->weight || !a->output) return TNX_E_INVALID;
  // 16-bit elements are read and written as such
  if (((uintptr_t)a->input & 1) || ((uintptr_t)a->weight & 1) || ((uintptr_t)a->output & (a->out_f32 ? 3 : 1))) return TNX_E_INVALID;
  if (a->bias && ((uintptr_t)a->bias & (a->bias_dtype == TNX_F32 ? 3 : 1))) return TNX_E_INVALID;
  unsigned grid = 0;
  hipError_t err;
  if (r.gemm) {
    tnx_gemm_args g;
    GemmBatch x;
    fill_gemm(a, r, &g, &x);
    return gemm_launch(&g, &x);
  }
  if (r.dma) {
    GemmParams p;
    fill_dma(a, r, &p, &grid);
    err = r.dma->conv(p, grid, (hipStream_t)a->stream);
  } else {
    ConvParams p;
    fill_registers(a, r, &p, &grid);
    err = r.reg->launch(p, grid, (hipStream_t)a->stream);
  }
  if (err != hipSuccess) {
    note_hip_error((int)err);
    return TNX_E_HIP;
  }
  return TNX_OK;
}

// register-staged tiles first, then the GEMM kernel's conv2d variants
template <class F> static void each_conv_kernel(F f) {
  int ng = 0;
  const ConvGroup* g = tnx_conv_groups(&ng);
  for (int i = 0; i < ng; ++i)
    for (int j = 0; j < g[i].count; ++j) f(g[i].entries[j].dtype, g[i].entries[j].block_cout, g[i].entries[j].block_pix, g[i].entries[j].block_k, false);
  const KernelGroup* k = tnx_kernel_groups(&ng);
  for (int i = 0; i < ng; ++i)
    for (int j = 0; j < k[i].count; ++j)
      if (k[i].entries[j].conv && find_dma(k[i].entries[j].dtype, k[i].entries[j].bm, k[i].entries[j].bn, k[i].entries[j].bk) == &k[i].entries[j])
        f(k[i].entries[j].dtype, k[i].entries[j].bm, k[i].entries[j].bn, k[i].entries[j].bk, true);
}

extern "C" int tnx_conv2d_kernel_count(void) {
  int n = 0;
  each_conv_kernel([&](int, int, int, int, bool) { ++n; });
  return n;
}

extern "C" const char* tnx_conv2d_kernel_name(int idx) {
  static thread_local char buf[64];
  int n = 0;
  buf[0] = 0;
  each_conv_kernel([&](int dtype, int bc, int bp, int bk, bool dma) {
    if (n++ == idx) snprintf(buf, sizeof buf, "%s %d %d %d %s", dtype == TNX_F16 ? "f16" : "bf16", bc, bp, bk, dma ? "dma" : "registers");
  });
  return buf;
}
