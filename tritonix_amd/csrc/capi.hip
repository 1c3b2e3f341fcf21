// C ABI of libtritonix_hip.so: argument checking, tile-kernel lookup, launch.
// Declarations and the reference interfaces they replace: include/tritonix_hip.h
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <string.h>

#include <cmath>
#include <mutex>
#include <unordered_map>

#include "../../include/tritonix_hip.h"
#include "registry.h"

using namespace tnx;

extern "C" const KernelGroup* tnx_kernel_groups(int* ngroups);  // generated

static thread_local int g_last_hip_error = 0;
namespace tnx {
void note_hip_error(int err) { g_last_hip_error = err; }
}

static int elem_size(int dt) { return dt == TNX_I8 ? 1 : (dt == TNX_F16 || dt == TNX_BF16) ? 2 : 4; }

// (by hash: walking the 315 entries took a third of a microsecond, twice per call)
static uint64_t entry_key(int dtype, int bm, int bn, int bk, int nw, int stages) {
  return ((((((uint64_t)dtype << 10 | (unsigned)bm) << 10 | (unsigned)bn) << 10 | (unsigned)bk) << 8 | (unsigned)nw) << 8) | (unsigned)stages;
}
static const KernelEntry* find_entry(const tnx_gemm_args* a) {
  static const std::unordered_map<uint64_t, const KernelEntry*> entries = [] {
    std::unordered_map<uint64_t, const KernelEntry*> m;
    int ng = 0;
    const KernelGroup* g = tnx_kernel_groups(&ng);
    for (int i = 0; i < ng; ++i)
      for (int j = 0; j < g[i].count; ++j) {
        const KernelEntry& e = g[i].entries[j];
        m.emplace(entry_key(e.dtype, e.bm, e.bn, e.bk, e.nw, e.stages), &e);
      }
    return m;
  }();
  if (a->block_m > 512 || a->block_n > 512 || a->block_k > 512 || a->num_warps > 64 || a->num_stages > 64 || a->block_m <= 0 ||
      a->block_n <= 0 || a->block_k <= 0 || a->num_warps <= 0 || a->num_stages <= 0 || a->in_dtype < 0)
    return nullptr;
  const auto hit = entries.find(entry_key(a->in_dtype, a->block_m, a->block_n, a->block_k, a->num_warps, a->num_stages));
  return hit == entries.end() ? nullptr : hit->second;
}


// LDS bytes of a tile config, whether or not a kernel is built for it
static bool is_skinny_cfg(const tnx_gemm_args* a) {
  return a->block_m == SKINNY_BM && a->block_n == SKINNY_BN && a->block_k == SKINNY_BK && a->num_warps == SKINNY_NW;
}

static int64_t lds_bytes_of(const tnx_gemm_args* a) {
  if (a->block_m <= 0 || a->block_n <= 0 || a->block_k <= 0 || a->num_stages <= 0) return -1;
  if (is_skinny_cfg(a)) return (int64_t)a->num_stages * SKINNY_NW * SKINNY_STEP_BYTES;
  int es = elem_size(a->in_dtype);
  const int64_t ring = (int64_t)a->num_stages * ((int64_t)a->block_m * a->block_k + (int64_t)a->block_k * a->block_n) * es;
  // the epilogue passes the accumulators through per-wave LDS strips laid over the ring (EpiStage in
  // gemm_tile.h): waves x MFMA rows x (wave-tile width x 4 bytes + 16).  Same wave grid as TileCfg.
  const int nw = a->num_warps > 0 ? a->num_warps : 4;
  const int wgm = nw == 4 ? 2 : (a->block_m > a->block_n ? 4 : 2), wgn = nw / wgm > 0 ? nw / wgm : 1;
  const int wtm = a->block_m / wgm, wtn = a->block_n / wgn;
  const int mi = 16;   // TileCfg::MI
  const int rows = mi;   // EpiStage::ROWS
  (void)wtm;
  const int64_t strips = (int64_t)nw * rows * (wtn * 4 + 16);
  // the persistent kernel keeps its (smaller) strips beside the ring: MI rows of 256 bytes per wave
  if (a->schedule & TNX_SCHED_PERSISTENT) return ring + (int64_t)nw * mi * 256;
  return ring > strips ? ring : strips;
}

static int check_common(const tnx_gemm_args* a, GemmForm form) {
  const bool pair = form == GEMM_PAIR;
  if (!a) return TNX_E_INVALID;
  if (a->m < 0 || a->n < 0 || a->k < 0) return TNX_E_INVALID;
  if (a->in_dtype != TNX_F16 && a->in_dtype != TNX_BF16 && a->in_dtype != TNX_I8 && !(form == GEMM_F32 && a->in_dtype == TNX_F32))
    return TNX_E_INVALID;
  if (a->epilogue < TNX_EPI_NONE || a->epilogue > TNX_EPI_GLU_IDENTITY) return TNX_E_INVALID;
  if (a->block_m <= 0 || a->block_n <= 0 || a->block_k <= 0 || a->group_m <= 0 || a->split_k <= 0 ||
      a->num_stages <= 0 || a->num_warps <= 0 || a->tail_tiles < 0 || a->schedule < 0 ||
      a->schedule > (TNX_SCHED_PERSISTENT | TNX_SCHED_SUPERBLOCK | TNX_SCHED_ATOMIC_REDUCE))
    return TNX_E_INVALID;
  // output type is tied to the input type: f16->f16, bf16->bf16, i8->i32
  // ... or binary32 for the 16-bit float types, on the tiles that carry that epilogue (f32_out_tile in gemm_tile.h)
  int want_out = a->in_dtype == TNX_I8 ? TNX_I32 : a->in_dtype;
  if (a->out_dtype != want_out) {
    const bool f32_out = a->out_dtype == TNX_F32 && a->in_dtype != TNX_I8 &&
                         ((int64_t)a->block_m * a->block_n <= 128 * 128 || pair) &&
                         !(a->schedule & TNX_SCHED_PERSISTENT) && !is_skinny_cfg(a);
    if (!f32_out) return TNX_E_UNSUPPORTED;
  }
  if (a->epilogue != TNX_EPI_NONE && (a->in_dtype == TNX_I8 || (a->n & 1))) return TNX_E_UNSUPPORTED;
  if (a->m > 0x7fffffff || a->n > 0x7fffffff || a->k > 0x7fffffff) return TNX_E_UNSUPPORTED;
  return TNX_OK;
}

// Which DMA loader the operands can take.  0: none, the element-wise loader only; 1: A and B row-major; 2: row-major A,
// k-contiguous B (stride_bk == 1, the layout of x @ w.t()); 3: m-contiguous A (stride_am == 1, x.t() @ dy), row-major B
// (only in the tiles built for it).  All want 16-byte aligned rows and base pointers, k % block_k == 0 and rows of whole
// 16-byte chunks.
// *tail: the operands have such a layout but not as the DMA loader likes it best -- K no multiple of block_k, rows or
// base pointers not 16-byte aligned (the loads take any byte address: probed on the hardware), N (layout 3: or M) ending
// inside a 16-byte chunk -- so the last K slab, the only one whose chunks can cross the end of a row of A or of the last
// row of B, is left out of the ring and fetched after it (GemmParams::tail_slab).  That fetch reads into what follows a row, so
// it needs a pitch of at least the row's length.
// *narrow: the operands have such a layout, but rows shorter than a chunk and a last slab of few rows let a chunk of the
// slab before it end past the operand (ring_chunks_inside): the layout is not taken.
static int dma_layout(const tnx_gemm_args* a, bool* tail = nullptr, bool* narrow = nullptr) {
  const int es = elem_size(a->in_dtype);
  const int vec = 16 / es;
  if (tail) *tail = false;
  if (narrow) *narrow = false;
  const int64_t last_rows = a->k > 0 && a->block_k > 0 ? (a->k - 1) % a->block_k + 1 : 0;      // k rows of the last slab
  const bool b_inside = ring_chunks_inside(last_rows, a->n, a->stride_bk, vec);
  if (a->stride_am == 1 && a->stride_ak != 1 && a->stride_bn == 1 && a->k > 0 && a->stride_ak >= a->m && a->stride_bk >= a->n &&
      (int64_t)a->block_k * a->stride_ak * es + (int64_t)a->block_m * es < (1ll << 32) &&
      (int64_t)a->block_k * a->stride_bk * es + (int64_t)a->block_n * es < (1ll << 32)) {
    const bool aligned = (a->stride_ak * es) % 16 == 0 && (a->stride_bk * es) % 16 == 0 && !((uintptr_t)a->a & 15) && !((uintptr_t)a->b & 15);
    if (aligned && a->k % a->block_k == 0 && a->m % vec == 0 && a->n % vec == 0) return 3;
    if (tail) {
      if (!b_inside || !ring_chunks_inside(last_rows, a->m, a->stride_ak, vec)) {
        if (narrow) *narrow = true;
        return 0;
      }
      *tail = true;
      return 3;
    }
  }
  if (a->stride_ak != 1 || a->k == 0 || a->stride_am < 0) return 0;
  // per-lane DMA offsets are 32-bit
  if ((int64_t)a->block_m * a->stride_am * es >= (1ll << 32)) return 0;
  const bool a_aligned = (a->stride_am * es) % 16 == 0 && !((uintptr_t)a->a & 15) && !((uintptr_t)a->b & 15);
  if (a->stride_bn == 1 && a->stride_bk >= 0 &&
      (int64_t)a->block_k * a->stride_bk * es + (int64_t)a->block_n * es < (1ll << 32)) {
    const bool strict = a_aligned && a->k % a->block_k == 0 && (a->stride_bk * es) % 16 == 0 && a->n % vec == 0 && a->n >= vec;
    if (strict) return 1;
    const bool loose_ok = tail && a->stride_am >= a->k && a->stride_bk >= a->n;
    if (loose_ok && b_inside) {
      *tail = true;
      return 1;
    }
    if (loose_ok && narrow) *narrow = true;
  }
  if (a->stride_bk == 1 && a->stride_bn >= 0 && (int64_t)a->block_n * a->stride_bn * es + (int64_t)a->block_k * es < (1ll << 32)) {
    if (a_aligned && a->k % a->block_k == 0 && (a->stride_bn * es) % 16 == 0) return 2;
    // the same relaxation for a k-contiguous B: rows of B^T at any alignment, any K
    if (tail && a->stride_am >= a->k && a->stride_bn >= a->k) {
      *tail = true;
      return 2;
    }
  }
  return 0;
}
extern "C" int64_t tnx_gemm_lds_bytes(const tnx_gemm_args* a) {
  if (!a) return -1;
  return lds_bytes_of(a);
}

// tiles that are cut along K: all of them, or the last tail_tiles in launch order
static int64_t cut_tiles(const tnx_gemm_args* a) {
  if (a->block_m <= 0 || a->block_n <= 0) return 0;
  int64_t tiles = ((a->m + a->block_m - 1) / a->block_m) * ((a->n + a->block_n - 1) / a->block_n);
  if (a->split_k <= 1) return 0;
  return a->tail_tiles > 0 && a->tail_tiles < tiles ? a->tail_tiles : tiles;
}

extern "C" size_t tnx_gemm_workspace_bytes(const tnx_gemm_args* a) {
  if (!a || a->split_k <= 1 || a->m <= 0 || a->n <= 0) return 0;
  if (is_skinny_cfg(a)) return 0;   // the eight K slices meet in LDS
  // every slice of a cut tile is kept whole (block_m x block_n accumulators of 4 bytes)
  return (size_t)WS_COUNTER_BYTES + (size_t)a->split_k * (size_t)cut_tiles(a) * (size_t)a->block_m * (size_t)a->block_n * 4;
}

// a tile that is built with the element-wise loader, for this problem's type and rows (null: none built)
static const KernelEntry* elementwise_tile(const tnx_gemm_args* a) {
  int ng = 0;
  const KernelGroup* g = tnx_kernel_groups(&ng);
  const KernelEntry* best = nullptr;
  for (int i = 0; i < ng; ++i)
    for (int j = 0; j < g[i].count; ++j) {
      const KernelEntry& e = g[i].entries[j];
      if (e.dtype != a->in_dtype || !e.generic || e.bm * e.bn > 128 * 128) continue;
      if (!best || (a->m <= 64 ? e.bm < best->bm : e.bm > best->bm)) best = &e;
    }
  return best;
}

static int supported_impl(const tnx_gemm_args* a, const KernelEntry** out, bool* fast, bool inspect_ptrs, bool* bt = nullptr,
                          bool* tail = nullptr, bool* at = nullptr, GemmForm form = GEMM_PLAIN, bool* other_tile = nullptr) {
  if (bt) *bt = false;
  if (at) *at = false;
  if (tail) *tail = false;
  if (other_tile) *other_tile = false;
  int st = check_common(a, form);
  if (st != TNX_OK) return st;
  int64_t lds = lds_bytes_of(a);
  if (lds > TNX_LDS_LIMIT_BYTES) return TNX_E_LDS;
  if (is_skinny_cfg(a)) {
    // m <= 16 rows, K cut eight ways inside the workgroup, DMA loader only
    if (a->split_k != SKINNY_SPLIT || a->epilogue != TNX_EPI_NONE || a->in_dtype == TNX_I8) return TNX_E_UNSUPPORTED;
    if (!skinny_lookup(a->in_dtype, a->num_stages)) return TNX_E_UNSUPPORTED;
    if (a->m > SKINNY_BM || a->m < 1 || a->n % SKINNY_BN != 0 || a->k % (SKINNY_SPLIT * SKINNY_BK) != 0 || a->k == 0)
      return TNX_E_UNSUPPORTED;
    if (a->stride_ak != 1 || a->stride_bn != 1 || (a->stride_am * 2) % 16 != 0 || (a->stride_bk * 2) % 16 != 0 ||
        a->stride_am < 0 || a->stride_bk < 0)
      return TNX_E_UNSUPPORTED;
    if (inspect_ptrs && ((((uintptr_t)a->a) & 15) || (((uintptr_t)a->b) & 15))) return TNX_E_UNSUPPORTED;
    if ((int64_t)SKINNY_BK * a->stride_bk * 2 >= (1ll << 32) || (int64_t)SKINNY_BM * a->stride_am * 2 >= (1ll << 32))
      return TNX_E_UNSUPPORTED;
    if (out) *out = nullptr;
    if (fast) *fast = true;
    return TNX_OK;
  }
  const KernelEntry* e = find_entry(a);
  if (!e) return TNX_E_UNSUPPORTED;
  tnx_gemm_args tmp = *a;
  if (!inspect_ptrs) { tmp.a = nullptr; tmp.b = nullptr; }
  const bool padded = form == GEMM_PADDED || form == GEMM_PAIR;
  if (padded) { tmp.m = (tmp.m + 7) / 8 * 8; tmp.n = (tmp.n + 7) / 8 * 8; }    // 16-bit operands: chunks of 8 elements
  bool tail_slab = false, narrow = false;
  // the persistent kernel keeps the strict layout
  const int layout = dma_layout(&tmp, (a->schedule & TNX_SCHED_PERSISTENT) ? nullptr : &tail_slab, &narrow);
  if (form == GEMM_PAIR && (a->out_dtype != TNX_F32 || layout == 0 || tail_slab || !e->pair[layout - 1])) return TNX_E_UNSUPPORTED;
  bool f = layout == 1 || (layout == 2 && e->fast_bt) || (layout == 3 && e->fast_at);
  if (tail) *tail = f && tail_slab;
  if (!f && narrow && !e->generic && (a->stride_ak == 1 || e->fast_at) && elementwise_tile(a)) {
    if (other_tile) *other_tile = true;             // gemm_launch runs it on that tile
  } else if (!f && !e->generic) {
    return TNX_E_UNSUPPORTED;
  }
  if (a->schedule & TNX_SCHED_PERSISTENT) {
    if (!e->persist || layout != 1 || a->split_k != 1 || a->k < (int64_t)a->num_stages * a->block_k) return TNX_E_UNSUPPORTED;
  }
  if (bt) *bt = f && layout == 2;
  if (at) *at = f && layout == 3;
  int64_t tiles = ((a->m + a->block_m - 1) / a->block_m) * ((a->n + a->block_n - 1) / a->block_n);
  if (tiles * a->split_k > 0x7fffffffll) return TNX_E_UNSUPPORTED;
  if (cut_tiles(a) > WS_MAX_TILES) return TNX_E_UNSUPPORTED;  // one arrival counter per cut tile
  if (tnx_gemm_workspace_bytes(a) >= (1ull << 32)) return TNX_E_UNSUPPORTED;  // slices are addressed with 32-bit offsets
  if (out) *out = e;
  if (fast) *fast = f;
  return TNX_OK;
}

// CUs of the current device (the persistent kernel launches one workgroup per CU); looked up once per device
static int compute_units(int* out) {
  static int cached[64];
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) { g_last_hip_error = (int)err; return TNX_E_HIP; }
  if (dev < 0 || dev >= 64) return TNX_E_UNSUPPORTED;
  if (!cached[dev]) {
    int n = 0;
    err = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    if (err != hipSuccess || n <= 0) { g_last_hip_error = (int)err; return TNX_E_HIP; }
    cached[dev] = n;
  }
  *out = cached[dev];
  return TNX_OK;
}

extern "C" int tnx_gemm_supported(const tnx_gemm_args* a) { return supported_impl(a, nullptr, nullptr, false); }

extern "C" int tnx_gemm_tail_slabs(const tnx_gemm_args* a) {
  bool fast = false, tail = false;
  const int st = supported_impl(a, nullptr, &fast, true, nullptr, &tail);
  return st != TNX_OK ? -1 : !fast ? (int)((a->k + a->block_k - 1) / a->block_k) : tail ? 1 : 0;
}

extern "C" int tnx_gemm(const tnx_gemm_args* a) { return tnx::gemm_launch(a, nullptr); }

bool tnx::gemm_tile_for(int dtype, int bm, int bn, int bk, int* num_warps, int* num_stages) {
  int ng = 0;
  const KernelGroup* g = tnx_kernel_groups(&ng);
  const KernelEntry* best = nullptr;
  for (int i = 0; i < ng; ++i)
    for (int j = 0; j < g[i].count; ++j) {
      const KernelEntry& e = g[i].entries[j];
      if (e.dtype != dtype || e.bm != bm || e.bn != bn || e.bk != bk || !e.fast || e.bm * e.bn > 128 * 128) continue;
      // Eight waves and two ring slots first, then the shallowest ring: these problems stream their operands once
      // through a short K loop, and what hides the latency of a tile's first slab and of its stores is more waves and a
      // second workgroup on the CU, not a deeper ring (measured on GEMMs shaped like the 1x1 layers of a ResNet-50:
      // 128x128x64 with 8 waves / 2 slots 39 us, 4 / 2 43 us, 4 / 3 75 us on [512 x 256] x [256 x 100352])
      // A 64x64 tile is too little work for eight waves: four waves and three slots there (measured on the small
      // layers, 2048 -> 512 channels at 7x7: 16.3 against 21.9 us).
      auto score = [](const KernelEntry& k) {
        const bool small = k.bm * k.bn <= 64 * 64;
        return (k.nw == (small ? 4 : 8) ? 100 : 0) + (k.stages == (small ? 3 : 2) ? 50 : 0) - k.stages;
      };
      if (!best || score(e) > score(*best)) best = &e;
    }
  if (!best) return false;
  *num_warps = best->nw;
  *num_stages = best->stages;
  return true;
}

// any_base: whatever the base pointers are (as if they were off 16 bytes, which refuses rows that overlap).
bool tnx::gemm_f32_direct(const tnx_gemm_args* a, bool any_base) {
  if (!a || a->in_dtype != TNX_F32 || a->k <= 0) return false;
  tnx_gemm_args t = *a;
  if (any_base) t.a = t.b = (const void*)4;
  const KernelEntry* e = nullptr;
  return supported_impl(&t, &e, nullptr, true, nullptr, nullptr, nullptr, GEMM_F32) == TNX_OK && e;
}

void tnx::gemm_tile_layouts(const tnx_gemm_args* a, bool* pair, bool* bt, bool* at) {
  const KernelEntry* e = find_entry(a);
  *pair = e && e->pair[0];
  *bt = e && (*pair ? e->pair[1] : e->fast_bt);
  *at = e && (*pair ? e->pair[2] : e->fast_at);
}

int tnx::gemm_check(const tnx_gemm_args* a, GemmForm form) {
  const int st = supported_impl(a, nullptr, nullptr, true, nullptr, nullptr, nullptr, form);
  if (st != TNX_OK) return st;
  const size_t need = tnx_gemm_workspace_bytes(a);
  return need > 0 && (!a->workspace || a->workspace_bytes < need || ((uintptr_t)a->workspace & 255)) ? TNX_E_WORKSPACE : TNX_OK;
}

int tnx::gemm_launch(const tnx_gemm_args* a, const GemmBatch* extra, GemmForm form) {
  const KernelEntry* e = nullptr;
  bool fast = false, bt = false, at = false, tail_slab = false, other_tile = false;
  int st = supported_impl(a, &e, &fast, true, &bt, &tail_slab, &at, form, &other_tile);
  if (st != TNX_OK) return st;
  if (extra && (form == GEMM_PAIR || e->bm * e->bn > 128 * 128 || a->split_k != 1 || (a->schedule & TNX_SCHED_PERSISTENT) || is_skinny_cfg(a) || extra->batch < 1 ||
                a->epilogue != TNX_EPI_NONE || (extra->bias && a->in_dtype == TNX_I8)))
    return TNX_E_UNSUPPORTED;
  if (!a->a || !a->b || !a->c) {
    if (a->m == 0 || a->n == 0) return TNX_OK;
    if (!a->c || (a->k > 0 && (!a->a || !a->b))) return TNX_E_INVALID;
  }
  if (a->m == 0 || a->n == 0) return TNX_OK;
  if (tnx_gemm_workspace_bytes(a) > 0 &&
      (!a->workspace || a->workspace_bytes < tnx_gemm_workspace_bytes(a) || ((uintptr_t)a->workspace & 255)))
    return TNX_E_WORKSPACE;
  if (other_tile) {
    const KernelEntry* x = elementwise_tile(a);
    tnx_gemm_args t = *a;
    t.block_m = x->bm; t.block_n = x->bn; t.block_k = x->bk; t.num_warps = x->nw; t.num_stages = x->stages;
    t.split_k = 1; t.tail_tiles = 0; t.schedule = TNX_SCHED_DEFAULT;
    return gemm_launch(&t, extra, form);
  }

  const int es_out = elem_size(a->out_dtype);
  GemmParams p;
  memset(&p, 0, sizeof(p));
  p.a = (const uint8_t*)a->a;
  p.b = (const uint8_t*)a->b;
  p.c = (uint8_t*)a->c;
  p.ws = (uint8_t*)a->workspace;
  p.m = a->m; p.n = a->n; p.k = a->k;
  p.sam = a->stride_am; p.sak = a->stride_ak;
  p.sbk = a->stride_bk; p.sbn = a->stride_bn;
  p.scm = a->stride_cm; p.scn = a->stride_cn;
  p.tiles_m = (int)((a->m + a->block_m - 1) / a->block_m);
  p.tiles_n = (int)((a->n + a->block_n - 1) / a->block_n);
  p.group_m = a->group_m;
  p.split_k = a->split_k;
  const int64_t ncut = cut_tiles(a);
  p.split_tile0 = a->split_k > 1 ? (int)((int64_t)p.tiles_m * p.tiles_n - ncut) : 0;
  int kt_total = (int)((a->k + a->block_k - 1) / a->block_k);
  p.ktiles_per_split = (kt_total + a->split_k - 1) / a->split_k;
  p.epilogue = a->epilogue;
  p.out_dtype = a->out_dtype;
  p.b_once = p.tiles_m == 1;
  p.tile_order = (a->schedule & TNX_SCHED_SUPERBLOCK) && a->split_k == 1 ? 1 : 0;
  p.atomic_reduce = (a->schedule & TNX_SCHED_ATOMIC_REDUCE) && a->split_k > 1 ? 1 : 0;
  p.c_vec_ok = a->stride_cn == 1 && ((a->stride_cm * es_out) % 16) == 0 && (((uintptr_t)a->c) % 16) == 0;
  p.c_row_ok = a->stride_cn == 1;
  p.tail_slab = tail_slab ? 1 : 0;
  const bool padded = form == GEMM_PADDED || form == GEMM_PAIR;
  p.m_load = padded ? (a->m + 7) / 8 * 8 : a->m;
  p.n_load = padded ? (a->n + 7) / 8 * 8 : a->n;
  int64_t problems = 1;
  if (extra) {
    p.batch = extra->batch;
    p.b_batch_bytes = extra->b_batch_bytes;
    p.c_batch_bytes = extra->c_batch_bytes;
    p.cv.bias = (const uint8_t*)extra->bias;
    p.cv.bias_dtype = extra->bias_dtype;
    problems = extra->batch;
    if ((int64_t)p.tiles_m * p.tiles_n * problems > 0x7fffffffll) return TNX_E_UNSUPPORTED;
  }

  hipStream_t stream = (hipStream_t)a->stream;
  hipError_t err;
  if (is_skinny_cfg(a)) {
    err = skinny_lookup(a->in_dtype, a->num_stages)(p, (unsigned)(a->n / SKINNY_BN), stream);
  } else if (a->schedule & TNX_SCHED_PERSISTENT) {
    int cus = 0;
    const int st2 = compute_units(&cus);
    if (st2 != TNX_OK) return st2;
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
    err = e->persist(p, (unsigned)(tiles < cus ? tiles : cus), stream);
  } else {
    unsigned grid = a->split_k > 1 ? (unsigned)(p.split_tile0 + ncut * a->split_k) : (unsigned)((int64_t)p.tiles_m * p.tiles_n * problems);
    if (form == GEMM_PAIR)
      err = e->pair[at ? 2 : bt ? 1 : 0](p, grid, stream);
    else
      err = (at ? e->fast_at : bt ? e->fast_bt : fast ? e->fast : e->generic)(p, grid, stream);
  }
  if (err != hipSuccess) { g_last_hip_error = (int)err; return TNX_E_HIP; }

  return TNX_OK;
}

// ---------------------------------------------------------------------------
// tnx_gemm_static_workspace: the split-K scratch lives in a file-scope device array instead of a
// caller-provided workspace, so the call allocates nothing.  `scratch` is a host-side handle here:
// the device address is looked up once per device with hipGetSymbolAddress and only that pointer
// is ever handed to kernels.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[TNX_STATIC_WORKSPACE_BYTES];

static constexpr int MAX_DEVICES = 64;
static void* g_scratch_ptr[MAX_DEVICES];
static std::mutex g_scratch_mutex;

__global__ void zero_words_kernel(int* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// device address of this device's copy of `scratch` (each GPU holds its own copy at its own address)
static int scratch_of_current_device(void** out) {
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) { g_last_hip_error = (int)err; return TNX_E_HIP; }
  if (dev < 0 || dev >= MAX_DEVICES) return TNX_E_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (err != hipSuccess || !ptr) { g_last_hip_error = (int)err; return TNX_E_HIP; }
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return TNX_OK;
}

extern "C" int tnx_gemm_static_workspace(const tnx_gemm_args* a) {
  if (!a) return TNX_E_INVALID;
  tnx_gemm_args t = *a;
  t.workspace = nullptr;
  t.workspace_bytes = 0;
  const size_t need = tnx_gemm_workspace_bytes(&t);
  if (need > 0) {
    if (need > (size_t)TNX_STATIC_WORKSPACE_BYTES) return TNX_E_STATIC_LIMIT;
    int st = supported_impl(&t, nullptr, nullptr, true);
    if (st != TNX_OK) return st;
    void* ptr = nullptr;
    st = scratch_of_current_device(&ptr);
    if (st != TNX_OK) return st;
    // The array keeps what the last call left.  The arrival counters of the tiles this launch cuts must
    // start at zero; a launch leaves them zero, but one that was aborted does not, so they are cleared
    // here with a small fill kernel (legal under graph capture, unlike a memset node).
    const int words = (int)cut_tiles(&t);
    hipLaunchKernelGGL(zero_words_kernel, dim3((words + 255) / 256), dim3(256), 0, (hipStream_t)t.stream, (int*)ptr, words);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) { g_last_hip_error = (int)err; return TNX_E_HIP; }
    if (t.schedule & TNX_SCHED_ATOMIC_REDUCE) {
      // The atomic reduction adds every slice into one copy behind the counters and needs that copy zero at
      // launch.  A launch of this kind leaves it zero, but the array may hold the slices of an earlier ordered
      // launch (or of another tile shape), so the copy this launch adds into is cleared first, same fill kernel.
      const int64_t sum_words = cut_tiles(&t) * (int64_t)t.block_m * t.block_n;   // < 2^23: need <= TNX_STATIC_WORKSPACE_BYTES
      hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((sum_words + 255) / 256)), dim3(256), 0, (hipStream_t)t.stream,
                         (int*)((unsigned char*)ptr + WS_COUNTER_BYTES), (int)sum_words);
      err = hipGetLastError();
      if (err != hipSuccess) { g_last_hip_error = (int)err; return TNX_E_HIP; }
    }
    t.workspace = ptr;
    t.workspace_bytes = TNX_STATIC_WORKSPACE_BYTES;
  }
  return tnx_gemm(&t);
}

// Modelled microseconds of a launch of one tile, fitted per tile and element size (16-bit, int8, float32).
//   start      launch, first slab and epilogue of a workgroup          turn    what every further workgroup on a CU adds
//   slab       a K slab of one workgroup per CU                        shared  a slab of as many as share a CU, against one
//   step       what part of such a round the first workgroup in it costs (the rest grows with their number)
//   crowd      slab's growth from few workgroups to one on every CU    bt      its growth for a k-contiguous B
//   a_off, b_off  ... for rows of A, of B that are not 16-byte aligned  tail    the last slab, where it is left out of the ring
//   cut, cut_slice, cut_all  K cut: fixed, per slice of 64 KiB, and per 16 MiB of slices in all
//   store      C, in units of 0.2 us per MB
struct TileCost {
  int bm, bn, nw, stages;
  double start, turn, slab, shared, step, crowd, cut, cut_slice, a_off, b_off, tail, store, cut_all, bt;
};
static const TileCost COST16[] = {
    {256, 256, 8, 2, 4.16, 0.00108, 1.18, 1.89, 0.746, 0.278, 2.83, 0.129, 0.11, 0.159, 2.8, 1.08, 4.01, 0},
    {256, 256, 4, 2, 7.61, 1.54, 1.17, 1.16, 0.703, 0.337, 2.5, 0.232, 0.144, 0.227, 5.69, 1.39, 3.89, 0},
    {256, 192, 8, 2, 4.16, 0.586, 0.929, 51.7, 0.739, 0.305, 2.53, 0.244, 0.152, 0.184, 2.69, 0.986, 3.57, 0.0163},
    {192, 256, 8, 2, 4.01, 0.785, 0.951, 44.5, 0.736, 0.305, 2.46, 0.248, 0.11, 0.205, 2.38, 0.85, 3.64, 0.0384},
    {192, 192, 8, 3, 4.54, 1.15, 0.621, 43.7, 0.712, 0.406, 2.59, 0.248, 0.134, 0.191, 2.08, 1.46, 3.9, 0.0314},
    {256, 128, 8, 3, 4.24, 0.735, 0.575, 5.24, 0.711, 0.439, 2.27, 0.257, 0.266, 0.164, 2.3, 1.14, 3.74, 0},
    {256, 128, 4, 3, 5.25, 1.57, 0.585, 7.21, 0.694, 0.399, 2.84, 0.206, 0.29, 0.224, 3.63, 1.21, 4, 0},
    {128, 256, 8, 3, 4.5, 1.7, 0.574, 17.8, 0.666, 0.442, 2.25, 0.389, 0.135, 0.231, 2.08, 0.845, 3.5, 0.00578},
    {128, 128, 8, 3, 3.91, 0.51, 0.356, 2.18, 0.752, 0.439, 1.73, 0.358, 0.196, 0.215, 1.32, 1.45, 4.14, 0},
    {128, 128, 8, 2, 3.12, 0.0154, 0.551, 0.877, 0.795, 0.356, 1.55, 0.351, 0.158, 0.186, 1.14, 1.33, 3.93, 0},
    {64, 256, 8, 3, 4.15, 1.62, 0.509, 3.44, 0.84, 0.0951, 2.1, 0.584, 0.131, 0.341, 1.14, 0.887, 3.96, 0},
    {128, 64, 8, 3, 3.42, 0.296, 0.298, 0.952, 0.875, 0.359, 1.26, 0.422, 0.267, 0.197, 0.911, 2.27, 5.21, 0},
    {64, 128, 8, 3, 3.63, 1.11, 0.328, 0.975, 0.896, 0.0551, 1.28, 0.648, 0.171, 0.3, 0.653, 1.35, 5.83, 0},
    {64, 128, 8, 4, 3.61, 1.22, 0.316, 0.6, 0.865, 0.052, 1.35, 0.633, 0.188, 0.327, 0.758, 1.28, 5.97, 0},
    {64, 64, 4, 4, 3.62, 0.794, 0.203, 0.493, 0.919, 0.308, 1.69, 0.884, 0.288, 0.366, 0.896, 0.0846, 2.06, 0},
    {32, 128, 4, 3, 3.81, 0.918, 0.259, 0.495, 0.874, 0.171, 1.73, 1.06, 0.127, 0.432, 0.983, 0.0198, 1.81, 0},
    {32, 64, 4, 4, 3.48, 0.431, 0.151, 1.1, 0.893, 0.276, 1.39, 1.51, 0.152, 0.472, 0.682, 0.103, 1.79, 0}};
static const TileCost COST8[] = {
    {256, 256, 8, 2, 4.92, 2.97, 1.16, 1.33, 0.673, 0.206, 2.71, 0.119, 0.141, 0.316, 2.63, 0.884, 3.56, 0.014},
    {256, 256, 4, 2, 8.13, 2.65, 1.16, 41.3, 33.4, 0.117, 2.41, 0.148, 0.182, 0.357, 4.58, 1.21, 4.01, 0.0384},
    {256, 192, 8, 2, 5.08, 3.12, 0.93, 45.5, 0.674, 0.228, 2.28, 0.209, 0.171, 0.325, 2.52, 0.785, 3.13, 0.00399},
    {192, 256, 8, 2, 4.56, 2.83, 0.93, 64, 0.74, 0.188, 2.06, 0.227, 0.13, 0.379, 2.43, 0.812, 3.65, 0.0327},
    {192, 192, 8, 3, 4.66, 2.92, 0.652, 42.1, 0.713, 0.309, 2.11, 0.328, 0.188, 0.323, 2.15, 0.927, 3.51, 0.0156},
    {256, 128, 8, 3, 4.26, 1.9, 0.621, 173, 0.698, 0.279, 1.78, 0.302, 0.29, 0.276, 2.04, 0.973, 3.52, 0.000823},
    {128, 256, 8, 3, 4.62, 2.87, 0.588, 16.7, 0.638, 0.326, 2.03, 0.414, 0.189, 0.387, 2.06, 0.807, 3.27, 0.0633},
    {128, 128, 8, 3, 3.7, 0.56, 0.377, 1.02, 0.917, 0.271, 1.47, 0.465, 0.303, 0.374, 1.42, 1.16, 4.28, 0},
    {128, 128, 8, 2, 3.25, 0.175, 0.498, 0.887, 0.757, 0.405, 1.36, 0.379, 0.253, 0.342, 1.39, 1.07, 4.12, 0},
    {64, 256, 8, 3, 4.09, 1.59, 0.477, 22.8, 0.853, 0.126, 1.47, 0.575, 0.198, 0.541, 1.52, 0.878, 4.04, 0.0117},
    {64, 128, 8, 3, 3.54, 1.24, 0.298, 0.883, 0.914, 0.175, 1.16, 0.614, 0.272, 0.453, 1.04, 0.996, 5.44, 0},
    {64, 128, 8, 4, 3.52, 1.28, 0.296, 0.6, 0.843, 0.128, 1.11, 0.623, 0.288, 0.477, 1.06, 1.04, 5.6, 0},
    {32, 128, 4, 3, 3.53, 0.276, 0.271, 0.628, 0.976, 0.00642, 1.1, 1.06, 0.264, 0.674, 1.18, 1.14, 4.32, 0}};
// ... of float32 operands as they are (TagF32)
static const TileCost COST32[] = {
    {64, 64, 4, 4, 3.78, 0.00146, 0.508, 0.815, 0.924, 0.00596, 1.19, 0.628, 0.0157, 0.0607, 0.611, 1.72, 5.8, 0},
    {32, 128, 4, 3, 4.29, 1.2, 0.535, 0.695, 0.752, 0.151, 1.58, 0.711, 0.0186, 0.0689, 0.782, 0.485, 1.38, 0},
    {32, 64, 4, 4, 3.68, 0.0338, 0.279, 1.48, 0.782, 0.133, 1.11, 1.04, 0.0341, 0.0867, 0.498, 1.33, 5.28, 0}};

// `s` slices of K, or as many as the same runs of slabs fill: kt = 81 cut in 10 is nine runs of nine, and the tenth slice would be a
// workgroup that stores a tile of zeros for the last one to read back.
static int filled_slices(int64_t kt, int s) {
  const int64_t per = (kt + s - 1) / s;
  return per > 0 ? (int)((kt + per - 1) / per) : 1;
}

struct Priced {
  int64_t m, n, kt, cus;
  bool a_off, b_off, ragged, bt;
  double c_mb, ab_mb;              // bytes of C, of A and B together, in MB
};
// s slices of K for every tile (tail 0) or for the last `tail` tiles
static double tile_time(const TileCost& t, const Priced& p, int s, int64_t tail) {
  const int64_t lds = (int64_t)(t.bm + t.bn) * 128 * t.stages, fit = TNX_LDS_LIMIT_BYTES / lds, most = t.nw == 8 ? 2 : 3;
  const int64_t c = fit < 1 ? 1 : fit < most ? fit : most;              // workgroups that share a CU
  const double cus = (double)p.cus, g = c > 1 ? 1.0 + t.shared : 1.0;
  const double slab = t.slab * (1.0 + (p.a_off ? t.a_off : 0.0)) * (1.0 + (p.b_off ? t.b_off : 0.0));
  auto of = [&](int64_t n) { return n <= 0 ? 0.0 : 1.0 + (g - 1.0) * (double)(n - 1) / (double)(c > 1 ? c - 1 : 1); };
  const double q = t.step < 1.0 ? t.step : 1.0;
  auto rounds = [&](int64_t groups, double slabs) {
    const int64_t full = groups / (p.cus * c), rem = groups - full * p.cus * c, n = (rem + p.cus - 1) / p.cus;
    const double fill = (double)groups / cus, frac = (double)rem / cus - (double)(n - 1);
    const double crowd = (groups <= p.cus ? 1.0 + t.crowd * fill * fill : 1.0 + t.crowd) * (p.bt ? 1.0 + t.bt : 1.0);
    double last = 0.0;
    if (rem > 0) last = n == 1 ? (full > 0 ? q + (1.0 - q) * frac : 1.0) : of(n - 1) + (of(n) - of(n - 1)) * (q + (1.0 - q) * frac);
    return (double)(full * c + n - 1) * t.turn + slab * slabs * crowd * ((double)full * g + last);
  };
  const int64_t tiles = ((p.m + t.bm - 1) / t.bm) * ((p.n + t.bn - 1) / t.bn), per = (p.kt + s - 1) / s;
  const double area = t.bm * t.bn / 16384.0;
  double us = tail > 0 ? rounds(tiles - tail, (double)p.kt) + t.turn + slab * (double)per * (1.0 + t.crowd) : rounds(tiles * s, (double)per);
  if (s > 1) us += t.cut + t.cut_slice * s * area + t.cut_all * (double)(tail > 0 ? tail : tiles) * s * area / 256.0;
  us += t.start + (p.ragged ? t.tail : 0.0) + t.store * p.c_mb / 5.0;
  const double stream = p.ab_mb / 6.0 + 2.0;
  return us > stream ? us : stream;
}

// The tile, its waves and slots, and the K cut with the smallest modelled time.  The constants are a least-squares fit of the
// logarithm to 273,000 launches: 3,979 problems of 17 to 8192 rows, 64 to 28672 columns and k of 64 to 14336 in bf16, f16
// and int8, nn, nt and tn, gated and not, odd sizes among them, on every tile here uncut and cut in 2 to 16, ten launches
// each in a graph.  Against the fastest of them the choice takes 1.021x the time in the mean (int8 1.027x), the one before
// (six tiles at fixed relative rates, cuts of 2, 4, 8 and 16 at 9 us each) 1.088x (int8 1.13x): on problems of 33 to 256 rows
// 0.88 to 0.90 of its time, to 1024 rows 0.94, above 0.96, int8 0.83 to 0.90; 4 % of the problems lose more than 5 %, 40 %
// gain more.  Slices are kept within what tnx_gemm_static_workspace holds (3136 x 1344 x 11632 with a k-contiguous B would want 35 MB
// of them: 102 us on 192x192 cut in two, 154 uncut).
// Three slabs of the 16-bit table are above the fit, by what 8,200 further problems measured: 128x64 by a tenth (column tiles of one row
// panel land on different L2s, which a tall A of long rows pays for: 3776 x 72 x 5952 16 -> 21 us where it took the place of 64x128),
// 64x256 by 4 % and 192x256 by 2 % (near ties with 128x128 and 256x256: 1024 x 13122 x 64 15 -> 21).  Of the choices that differ from
// the one before, 116 instead of 153 of 2,800 now lose 3 %, 29 instead of 51 lose 10 %.
// only_cut > 0: that many slices and no other number.
static double price_tiles(tnx_gemm_args* a, int es, bool at, int64_t cus, int only_cut = 0) {
  const int vec = 16 / es, bk = 128 / es;
  a->block_k = bk;
  Priced p;
  p.m = a->m; p.n = a->n; p.kt = (a->k + bk - 1) / bk; p.cus = cus;
  p.bt = a->stride_bk == 1 && a->stride_bn != 1;
  const int64_t ra = at ? a->stride_ak : a->stride_am, rb = p.bt ? a->stride_bn : a->stride_bk;
  p.a_off = ra % vec != 0 || ((uintptr_t)a->a & 15) != 0;
  p.b_off = rb % vec != 0 || ((uintptr_t)a->b & 15) != 0;
  p.ragged = p.a_off || p.b_off || a->k % bk != 0 || a->n % vec != 0;
  p.c_mb = (double)a->m * (double)(a->epilogue == TNX_EPI_NONE ? a->n : a->n / 2) * (es == 2 ? 2 : 4) * 1e-6;
  p.ab_mb = ((double)a->m + (double)a->n) * (double)a->k * es * 1e-6;
  const TileCost* table = es == 1 ? COST8 : es == 4 ? COST32 : COST16;
  const int type = a->in_dtype == TNX_I8 ? 2 : a->in_dtype == TNX_F16 ? 1 : a->in_dtype == TNX_F32 ? 3 : 0;
  static const int cuts[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16};
  struct Entries {                 // the kernels behind the tables (looking one up takes a third of a microsecond)
    const KernelEntry* of[4][sizeof COST16 / sizeof *COST16];
    int count[4];
    Entries() {
      static_assert(sizeof COST8 <= sizeof COST16 && sizeof COST32 <= sizeof COST16, "one array holds any table");
      for (int d = 0; d < 4; ++d) {
        count[d] = (int)((d == 3 ? sizeof COST32 : d == 2 ? sizeof COST8 : sizeof COST16) / sizeof *COST16);
        for (int i = 0; i < count[d]; ++i) {
          const TileCost& t = (d == 3 ? COST32 : d == 2 ? COST8 : COST16)[i];
          tnx_gemm_args q = {};
          q.in_dtype = d == 3 ? TNX_F32 : d == 2 ? TNX_I8 : d == 1 ? TNX_F16 : TNX_BF16;
          q.block_m = t.bm; q.block_n = t.bn; q.block_k = d == 3 ? 32 : d == 2 ? 128 : 64; q.num_warps = t.nw; q.num_stages = t.stages;
          of[d][i] = find_entry(&q);
        }
      }
    }
  };
  static const Entries entries;
  double best = 1e300;
  const TileCost* pick = nullptr;
  int best_s = 1, best_tail = 0;
  for (int i = 0; i < entries.count[type]; ++i) {
    const TileCost& t = table[i];
    // 256x256: two waves per SIMD cover the start and end of a short K loop, at half again as many LDS reads, which lose on the
    // long, power-limited ones (8192^3: 2 %; 4096 x 28672 x 4096, gated: 2.4 % the other way)
    if (t.bm == 256 && t.bn == 256 && t.nw != ((es == 2 && p.kt <= 64) || at ? 8 : 4)) continue;
    const KernelEntry* e = entries.of[type][i];
    if (!e || (at ? !e->fast_at : p.bt ? !e->fast_bt : !e->fast)) continue;
    const int64_t tiles = ((a->m + t.bm - 1) / t.bm) * ((a->n + t.bn - 1) / t.bn);
    if ((double)t.bm * t.bn * (double)tiles > 5.0 * (double)a->m * (double)a->n + 4.0 * 65536) continue;
    for (int cut : cuts) {
      if (only_cut > 0 && cut > 1) break;
      const int s = filled_slices(p.kt, only_cut > 0 ? only_cut : cut);
      const bool last_only = s > 1 && tiles > cus && tiles % cus != 0;         // only the tiles of the partial round are cut
      const int64_t tail = last_only ? tiles % cus : 0, ncut = s == 1 ? 0 : last_only ? tail : tiles;
      if (s > 1 && (p.kt / s < 2 || ncut > WS_MAX_TILES || ncut * s > (last_only ? 2 : 3) * cus ||
                    ncut * s * t.bm * t.bn * 4 > TNX_STATIC_WORKSPACE_BYTES - WS_COUNTER_BYTES))
        break;
      // (what is modelled to be even goes to the fewer slices: 4 % per doubling, 83 instead of 104 of 2,866 problems lose 5 %)
      const double us = tile_time(t, p, s, tail) * (1.0 + 0.04 * log2((double)s));
      if (us < best) { best = us; pick = &t; best_s = s; best_tail = (int)tail; }
    }
  }
  if (!pick) { a->block_m = 128; a->block_n = 128; a->num_stages = 3; a->num_warps = 8; return 1e300; }
  a->block_m = pick->bm; a->block_n = pick->bn; a->num_stages = pick->stages; a->num_warps = pick->nw;
  a->split_k = best_s; a->tail_tiles = best_tail;
  return best;
}

// large_f32: a problem of tnx_gemm_f32 (heads and tails in bf16), which may also go to the tiles of 192 and 256
static int default_config(tnx_gemm_args* a, bool large_f32);

extern "C" int tnx_gemm_default_config(tnx_gemm_args* a) {
  if (!a) return TNX_E_INVALID;
  if (a->in_dtype == TNX_F32) {
    // the bf16 problem tnx_gemm_f32 makes of it: heads and tails along k, aligned operands, k or the other dimension
    // contiguous as in the float32 operand
    tnx_gemm_args t = *a;
    t.in_dtype = TNX_BF16; t.out_dtype = TNX_F32;
    t.a = t.b = nullptr;
    t.m = (a->m + 7) / 8 * 8; t.n = (a->n + 7) / 8 * 8;
    t.k = (a->k + 31) / 32 * 64;
    const bool bt = a->stride_bk == 1 && a->stride_bn != 1, at = !bt && a->stride_am == 1 && a->stride_ak != 1 && a->stride_bk != 1;
    t.stride_am = at ? 1 : t.k; t.stride_ak = at ? t.m : 1;
    t.stride_bk = bt ? 1 : t.n; t.stride_bn = bt ? t.k : 1;
    const int st = default_config(&t, true);
    a->block_m = t.block_m; a->block_n = t.block_n; a->block_k = t.block_k; a->group_m = t.group_m;
    a->split_k = t.split_k; a->tail_tiles = t.tail_tiles; a->schedule = t.schedule;
    a->num_stages = t.num_stages; a->num_warps = t.num_warps;
    return st;
  }
  return default_config(a, false);
}

static int default_config(tnx_gemm_args* a, bool large_f32) {
  const int es = elem_size(a->in_dtype);
  const int bk = es == 1 ? 128 : 64;   // 128 bytes of K per LDS row for either element size
  // Workgroups that run together: the CU count of the current device, or MI355X's 256 when no device can be asked
  // (host-side planning).  The cost constants below are measured on MI355X.
  int64_t cus = 256;
  {
    int n = 0;
    if (compute_units(&n) == TNX_OK && n > 0) cus = n;
  }
  a->group_m = 8;
  a->split_k = 1;
  a->tail_tiles = 0;
  a->schedule = TNX_SCHED_DEFAULT;
  a->block_k = bk;
  bool dma_ok, at = false;
  {
    tnx_gemm_args t = *a;   // a and b, when given, count with their base alignment (null = aligned)
    if (t.stride_ak == 0 && t.stride_bn == 0) { t.stride_am = t.k; t.stride_ak = 1; t.stride_bk = t.n; t.stride_bn = 1; }
    t.block_m = 128; t.block_n = 128; t.block_k = bk;
    bool tail_slab = false;
    const int layout = dma_layout(&t, &tail_slab);
    dma_ok = layout != 0;     // every tile the choice below proposes is built for the DMA layouts ...
    at = layout == 3;         // ... except the 64-row int8 tiles, whose rows are too short to read an m-contiguous A from
  }
  if (a->m <= 64 && dma_ok && !(at && es == 1)) {
    // Skinny: B is streamed once, by at most one workgroup per CU, K cut further while that shortens the launch.
    // 16-bit types: 64 columns per workgroup keep the chip busy with half the K cuts that 128 need, and the hand-over of
    // the slices is a fixed cost per cut (16 x 4096 x 4096: 64 columns / 4 cuts 11.2 us, 128 / 8 12.7; 16 x 2048 x 4096
    // 8.7 against 11.8; 64 x 2048 x 4096 11.3 against 17.0).  With a row-major B the wider rows stream better once
    // there are enough bytes to stream, or enough columns for one round without a cut (64 x 8192 x 14336: 47.4 us with
    // 128 columns, 52.9 with 64; 16 x 28672 x 4096: 38.5 against 44.1); rows of a k-contiguous B are k runs either way.
    // Cutting s -> 2s saves kt / 2s slabs of the loop and costs s more slices: it pays while kt >= 1.75 s^2 (fitted to
    // 51 shapes of bf16 and int8, n 1024 to 28672, k 1024 to 14336; kt / s >= 4 and up to 512 workgroups before: 1.14x in
    // the mean), once the loop is long enough to pay for the first cut's hand-over of 1.2 to 2.5 us: 18 slabs of the 16-bit
    // types, 12 of int8, 14 of heads and tails (1,020 shapes, 1 to 64 slabs: the choice 1.01x the best cut in the mean, 1.14x
    // with cuts from 2 slabs on; 48 x 4096 x 128 bf16 5.7 -> 3.9 us, 48 x 2048 x 384 int8 6.6 -> 4.6).  int8 of up to 16 rows
    // hands less over and cuts from 1.25 s^2 on (8 x 256 x 10240 with a k-contiguous B: 9.3 us with 8 cuts, 8.1 with 16).
    // A k-contiguous B whose slices are an odd multiple of 32 slabs takes one cut more: such slices are 4 KB runs, the
    // workgroups all read at the same offsets modulo 4 KB, and halving them spreads the reads (16 x 8192 x 4096 bf16 16.2 ->
    // 13.7 us, 16 x 4096 x 8192 16.4 -> 14.0, 16 x 12288 x 8192 int8 23.5 -> 20.7, 16 x 8192 x 6144 float32 113 -> 104; slices of
    // 16, 24, 48 or 64 slabs lose 2 to 14 %).  Uncut it gains for int8 alone (16 x 28672 x 4096 24.3 -> 21.9).
    // Up to 32 rows a 32-row tile (not built for an m-contiguous A or for heads and tails), except where 128
    // columns are cut: 16 x 4096 x 14336 24.1 us on 64 rows and eight waves, 24.7 on 32 and four.
    const int64_t kt = (a->k + bk - 1) / bk;
    const bool bt = a->stride_bk == 1 && a->stride_bn != 1;
    // (A k-contiguous B of 200 MB or more, where 128 columns leave half a round and K is cut: 16 x 16384 x 14336 91 us with 64
    // columns, 70 with 128; 16 x 12288 x 14336 75 against 60.  Heads and tails: where 64 columns are not cut and k is an odd
    // multiple of 4 KB, see above: 16 x 16384 x 3072 float32 112 us with 64 columns, 104 with 128 cut in two.)
    const bool wide_bt = (a->n + 127) / 128 * 2 <= cus &&
                         (large_f32 ? (a->n + 63) / 64 * 2 > cus && kt % 64 == 32 : a->n * a->k >= 96000000);
    const bool narrow = es == 2 && (bt ? !wide_bt : (a->n + 63) / 64 <= cus && a->n * a->k <= 40000000);
    a->block_n = narrow ? 64 : 128;
    const int64_t tiles = (a->n + a->block_n - 1) / a->block_n;
    int s = 1;
    if (kt >= (es == 1 ? 12 : large_f32 ? 14 : 18))
      while (tiles * s * 2 <= cus && s < 16 && 4 * kt >= (es == 1 && a->m <= 16 ? 5 : 7) * s * s) s *= 2;
    if (bt && s >= (es == 1 ? 1 : 2) && s < 8 && kt % (64 * s) == 32 * s) s *= 2;
    s = filled_slices(kt, s);
    a->split_k = s;
    a->block_m = es == 2 && a->m <= 32 && !at && !large_f32 && (narrow || s == 1) ? 32 : 64;
    a->num_stages = narrow ? 4 : 3;
    a->num_warps = narrow || a->block_m == 32 ? 4 : 8;
    // 33 to 64 rows: the tile by modelled time (two rounds of 32 rows, three of which share a CU, mostly: 64 x 3840 x 6272
    // 16.9 -> 14.1 us), the cut as above -- an m-contiguous A then gives the bits of its row-major copy (434 problems: 0.89
    // of the time of the tiles above, 0.85 with the best cut too)
    if (es == 2 && !large_f32 && a->out_dtype != TNX_F32 && !at && a->m > 32) {
      tnx_gemm_args t = *a;
      if (price_tiles(&t, es, at, cus, s) < 1e300) *a = t;
    }
    return TNX_OK;
  }
  if (a->m <= 64 && at) {
    // int8 of few rows and an m-contiguous A: 128 rows are the fewest that the transposing read takes, K cut by the rule
    // above with its own least length (16 x 4096 x 4096: 14.2 us uncut, 9.2 cut in 8; 48 x 8192 x 4096 15.9, 13.7 in 4; uncut up
    // to 15 slabs: 48 x 4096 x 1536 8.0, 9.0 in 4).  Copying such an A into rows first and taking the tiles above: 11.4, 16.0
    // and 11.8 us.
    a->block_m = 128; a->block_n = 128; a->num_stages = 3; a->num_warps = 8;
    const int64_t kt = (a->k + bk - 1) / bk, tiles = (a->n + 127) / 128;
    int s = 1;
    if (kt >= 16)
      while (tiles * s * 2 <= cus && s < 16 && 4 * kt >= 7 * s * s) s *= 2;
    a->split_k = filled_slices(kt, s);
    return TNX_OK;
  }
  // operands the DMA loader cannot take (not row-major with unit inner strides, int8 rows that are not 16-byte
  // aligned) go to one of the two tiles that are also built with the element-wise loader
  if (!dma_ok) {
    a->block_m = a->m <= 64 ? 64 : 128; a->block_n = 128; a->num_stages = 2; a->num_warps = 4;
    return TNX_OK;
  }
  // 16-bit and int8 results
  // (two rounds and more of 256x256 tiles with long K loops run against the power limit, which the rates below are from and the
  // fitted launches, ten in a row, hardly meet)
  const bool powered = ((a->m + 255) / 256) * ((a->n + 255) / 256) >= 2 * cus && a->k >= 64 * bk;
  if (!large_f32 && a->out_dtype != TNX_F32 && !powered) {
    price_tiles(a, es, at, cus);
    const int64_t tm = (a->m + a->block_m - 1) / a->block_m, tn = (a->n + a->block_n - 1) / a->block_n;
    if (a->split_k == 1 && tm >= 16 && tn >= 16) a->schedule = TNX_SCHED_SUPERBLOCK;
    return TNX_OK;
  }
  // those, and binary32 results: pick the tile and the K cut with the smallest modelled time.  A wave is 256 workgroups (one per CU); a tile
  // costs its multiply-adds over the rate a CU sustains with that tile (relative rates measured on 8192^3 and
  // 2048^2 x 8192: 256x256 1.0, 256x128 0.9, 128x128 0.75); a last, partial wave costs 0.75 of a full one (the
  // part is power-limited: fewer busy CUs clock higher; measured 0.70-0.80 on 6144^3, 5120^2 x 8192,
  // 4096 x 5120 x 4096).  Cutting K costs a hand-over: a fixed 9 us plus the slices the finishing workgroup
  // reads back at about 60 GB/s.  Three shapes of launch are priced per tile: uncut; every tile cut (only when
  // the tiles alone leave CUs idle); only the tiles of the partial wave cut (tail_tiles).  Slices never get
  // shorter than eight K slabs.
  // (the sixth, 192x192, exists for the 16-bit types: it is what divides sides like 1536, 3072 or 4608 into whole
  // rounds -- 3072^3 is 144 tiles of 256x256 on 256 CUs, and 256 of these: measured 62 -> 47 us)
  // (192x256 and 256x192 likewise: 4096 x 2560 x 8192 is 160 tiles of 256x256, 0.63 of a round, and 220 of 192x256:
  // measured 141 -> 128 us; their rate lies between what they reach against 256x256 on 8192^3, 0.86, and on
  // launches of a round or two at K = 4096, where they run at the full 0.75 of its tile time)
  static const int cand[][4] = {{256, 256, 2, 4}, {256, 128, 3, 4}, {128, 128, 3, 4}, {64, 128, 3, 4}, {64, 64, 4, 4}, {192, 192, 3, 8},
                                {192, 256, 2, 8}, {256, 192, 2, 8}};
  static const double rate[] = {1.0, 0.9, 0.75, 0.5, 0.35, 0.92, 0.9, 0.9};
  const int ncand = 8;
  // int8: rows of a 64-wide B tile are too short for the transposing read; the 192-wide tiles exist for it too
  // (3072 x 4096 x 4096: 53.6 -> 45.7 us with 192x256, 4096 x 3072 x 4096: 52.8 -> 47.3 us with 256x192)
  // (a binary32 result exists on the tiles up to 128x128 and, for float32 products, on the eight-wave tiles of 192 and 256)
  // (and only while a lane's 32-bit offset reaches from the first to the last of the tile's k-contiguous rows)
  auto reach = [&](int i) {
    return !large_f32 || ((at || cand[i][0] * a->k * 2 < (1ll << 32)) && (a->stride_bk != 1 || a->stride_bn == 1 || cand[i][1] * a->k * 2 < (1ll << 32)));
  };
  auto usable = [&](int i) { return reach(i) && (es == 2 || i != 4) && !(at && es == 1 && i == 3) && (a->out_dtype != TNX_F32 || (i >= 2 && i <= 4) || (large_f32 && i != 1)); };
  const double cu_flops = 5.5e12 * (es == 1 ? 1.7 : 1.0);          // per CU with the largest tile
  const double launch = 3e-6, handover = 9e-6, readback = 60e9;
  const int64_t kt = (a->k + bk - 1) / bk;
  double best = 1e300;
  int bi = es == 1 ? (at ? 2 : 3) : 4, bs = 1, btail = 0;
  auto offer = [&](double t, int i, int s, int tail) {
    if (t < best * 0.97) { best = t; bi = i; bs = s; btail = tail; }   // ties go to the earlier (larger, less cut) choice
  };
  // (The 0.75 holds for nearly full last waves of the large tiles too: 220 tiles of 192x256 on 256 CUs took 0.80 of a
  // full wave's time; a cost that rises with the fill, 0.7 + 0.3 * rem / 256, was tried on 382 shapes and moved a
  // third of 75 choices for the worse by up to 20 %.  The tiles up to 128x128 do not load the power limit, so their
  // partial wave runs no faster than a full one: 128 tiles of 64x128 took 0.91 of the modelled full wave where 256
  // tiles of 64x64 took 1.0 of theirs; they are priced at 0.9.)
  for (int i = 0; i < ncand; ++i) {
    if (!usable(i)) continue;
    const int64_t tiles = ((a->m + cand[i][0] - 1) / cand[i][0]) * ((a->n + cand[i][1] - 1) / cand[i][1]);
    const double tile_t = 2.0 * cand[i][0] * cand[i][1] * (double)a->k / (cu_flops * rate[i]);
    const double slice_bytes = (double)cand[i][0] * cand[i][1] * 4;
    const double part = (i >= 2 && i <= 4) ? 0.9 : 0.75;            // cost of a last, partial wave (see above)
    const int64_t full = tiles / cus, rem = tiles % cus;
    offer((double)full * tile_t + (rem ? part * tile_t : 0.0) + launch, i, 1, 0);
    for (int s = 2; s <= 16; s *= 2) {
      if (kt / s < 8) break;
      if (full == 0 && tiles * s <= cus)                             // every tile cut (one wave at most)
        offer(tile_t / s + handover + s * slice_bytes / readback + launch, i, s, 0);
      if (full > 0 && rem > 0 && rem * s <= cus)                     // only the partial wave cut
        offer((double)full * tile_t + tile_t / s + handover + s * slice_bytes / readback + launch, i, s, (int)rem);
    }
  }
  a->block_m = cand[bi][0]; a->block_n = cand[bi][1]; a->num_stages = cand[bi][2]; a->num_warps = cand[bi][3];
  // The 128x128 tile, and the 64x128 tile of the 16-bit types, run with eight waves: problems that end up on them are
  // a few rounds of short tiles, and two waves per SIMD hide more of a tile's start and end than one (measured on
  // fifteen bf16 shapes from 768x3072x768 to 1024x4096x4096, three ring slots both: 1-14 % faster on every one, e.g.
  // 2048^3 21.2 -> 19.6 us, 2048^2 x 512 9.4 -> 8.1 us, 1024^3 9.1 -> 7.9 us; int8 128x128 5-13 % on seven shapes,
  // int8 64x128 mixed).
  if (bi == 2 || (es == 2 && bi == 3)) a->num_warps = 8;
  // (float32 products run three MFMA steps on the fragments of two, so fewer fragment reads decide: four waves, 2048^3
  // 55.2 -> 54.1 us, 4096^3 333 -> 327 us; not for an m-contiguous A, whose transposing reads double the count: 57 us with
  // eight, above 71 with four.)
  if (bi == 2 && large_f32 && !at) a->num_warps = 4;
  // A k-contiguous B on 64x128 tiles, one workgroup per CU: a fourth slot (the LDS holds six; five and six measured no
  // better) covers the longer way of 128-byte runs.  launches back to back: 512 x 4096 x 4096 23.6 -> 20.9 us, 1024 x 2048 x 4096
  // 22.4 -> 20.1, 512 x 4096 x 2048 12.2 -> 11.2 (whole calls on changing operands, the first of them: 23.1 -> 21.2); with two
  // workgroups on a CU three slots stay ahead (2048^3: 21.3 against 23.2 us), and with a row-major B they tie.
  if (es == 2 && bi == 3 && !large_f32 && a->stride_bk == 1 && a->stride_bn != 1 &&
      ((a->m + 63) / 64) * ((a->n + 127) / 128) * bs <= cus)
    a->num_stages = 4;
  // 16-bit problems with a short K loop (at most 64 slabs per tile) spend a visible share of every tile outside
  // it; two waves per SIMD cover that better than one (measured on 4096 x 28672 x 4096, gated: +2.4 %), at the
  // price of half again as many LDS reads, which is what loses on the long, power-limited 8192^3 loops.
  // (cut tiles too: 4096 x 5120 x 4096 with its last 64 tiles cut, 155 -> 140 us)
  if (es == 2 && bi == 0 && kt <= 64) a->num_warps = 8;
  if (bi == 0 && a->out_dtype == TNX_F32) a->num_warps = 8;
  if (at && bi == 0) a->num_warps = 8;                               // the only 256x256 kernels built for an m-contiguous A
  a->split_k = filled_slices(kt, bs);
  a->tail_tiles = btail;
  // Grids of several rounds of 256 tiles in both directions: the super-block order keeps what one round reads
  // to 16 + 16 operand panels and lets consecutive rounds share half of them (measured on 8192^3: int8 +4 %,
  // bf16 unchanged on random operands -- that launch is limited by board power -- and +12 % on operands that
  // draw less power; never slower).  The persistent schedule is not chosen: measured 1-3 % slower on the
  // benchmark shapes (it gives up the dynamic hand-out of tiles to whichever CU is free).
  {
    const int64_t tm = (a->m + a->block_m - 1) / a->block_m, tn = (a->n + a->block_n - 1) / a->block_n;
    if (bs == 1 && tm >= 16 && tn >= 16) a->schedule = TNX_SCHED_SUPERBLOCK;
  }
  return TNX_OK;
}

// tnx_gemm_default_config for a float32 product, or a tile that multiplies its operands as they are (TagF32) instead of heads
// and tails where that is modelled to be faster.
// The binary32 instruction has a sixteenth of bf16's rate where the split takes three bf16 products, but the split reads both
// operands once more, writes and reads their terms, and is a launch of its own: up to 64 rows the direct product is ahead
// everywhere (16 x 10112 x 7616 with a k-contiguous B: 176 -> 55 us, 5 x 7664 x 4992 87 -> 31), and so is one of up to 3e8
// operations (7.0 -> 4.9 us); from 3e9 on and 256 rows the split.  Split: a pass at 0.39 us per MB of operands and 5.4 us of
// its own and the second launch, then rounds of workgroups; constants from 2,900 problems, on which the choice takes 0.71x the
// split's time in the mean and loses more than 5 percent on 24.  Its sums are closer to the float64 product (2e-7 to 2e-6)
// than the split's (5e-6).
extern "C" int tnx_gemm_f32_config(tnx_gemm_args* a) {
  if (!a || a->in_dtype != TNX_F32) return TNX_E_INVALID;
  const int st = tnx_gemm_default_config(a);
  if (st != TNX_OK) return st;
  const tnx_gemm_args split = *a;
  tnx_gemm_args t = *a;
  t.a = t.b = (const void*)4;               // whatever the base pointers will be
  if (t.stride_ak == 0 && t.stride_bn == 0) { t.stride_am = t.k; t.stride_ak = 1; t.stride_bk = t.n; t.stride_bn = 1; }
  t.block_m = 64; t.block_n = 128; t.block_k = 32;
  bool tail_slab = false;
  const int layout = t.k > 0 ? dma_layout(&t, &tail_slab) : 0;
  if (layout == 0) return TNX_OK;
  t.a = t.b = nullptr;
  int64_t cus = 256;
  int n = 0;
  if (compute_units(&n) == TNX_OK && n > 0) cus = n;
  t.group_m = 8; t.split_k = 1; t.tail_tiles = 0; t.schedule = TNX_SCHED_DEFAULT;
  const double direct = price_tiles(&t, 4, layout == 3, cus);
  const double kt = (double)((a->k + 31) / 32), s = split.split_k, area = split.block_m * split.block_n / 16384.0;
  const double tiles = (double)((a->m + split.block_m - 1) / split.block_m) * (double)((a->n + split.block_n - 1) / split.block_n);
  const double rounds = ceil(tiles * (split.tail_tiles ? 1.0 : s) / (double)cus), per = split.tail_tiles ? kt : ceil(kt / s);
  const double in_mb = ((double)a->m + (double)a->n) * (double)a->k * 4e-6, out_mb = (double)a->m * (double)a->n * 4e-6;
  const double both = 5.44 + 0.388 * in_mb + 0.337 * out_mb + rounds * (0.37 + per * (0.14 + 0.373 * area)) + (s > 1 ? 1.58 + 0.663 * s * area : 0.0);
  if (direct * 1.03 > both) return TNX_OK;
  a->block_m = t.block_m; a->block_n = t.block_n; a->block_k = t.block_k; a->group_m = t.group_m;
  a->split_k = t.split_k; a->tail_tiles = t.tail_tiles; a->schedule = t.schedule;
  a->num_stages = t.num_stages; a->num_warps = t.num_warps;
  return TNX_OK;
}

// ---------------------------------------------------------------------------
// float32 operands as bf16 head and tail (see tnx_split_f32 in the header)
// ---------------------------------------------------------------------------
__global__ void split_f32_kernel(const float* src, int64_t rows, int64_t cols, int64_t sr, int64_t sc, uint16_t* dst, int side) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * cols) return;
  const int64_t i = idx / cols, j = idx - i * cols;
  const float v = src[i * sr + j * sc];
  const __bf16 hi = (__bf16)v;                                        // round to nearest even
  const float rest = v - (float)hi;
  // An infinity or NaN lives in the head alone: its tail is zero, and so is the second copy of its head -- the one
  // that meets the other operand's tail -- or inf * (a tail that happens to be 0) would turn an infinite sum into NaN.
  const bool fin = __builtin_isfinite(rest) && __builtin_isfinite((float)hi);
  const __bf16 lo = fin ? (__bf16)rest : (__bf16)0.0f;
  const uint16_t h = __builtin_bit_cast(uint16_t, hi), l = __builtin_bit_cast(uint16_t, lo);
  const uint16_t h2 = fin ? h : (uint16_t)0;
  if (side == 0 || side == 2) {
    uint16_t* row = dst + i * 3 * cols;
    row[j] = h;
    row[cols + j] = side == 0 ? h2 : l;
    row[2 * cols + j] = side == 0 ? l : h2;
  } else {
    dst[i * cols + j] = h;
    dst[(rows + i) * cols + j] = l;
    dst[(2 * rows + i) * cols + j] = h2;
  }
}

extern "C" int tnx_split_f32(const float* src, int64_t rows, int64_t cols, int64_t stride_r, int64_t stride_c, void* dst, int side,
                             void* stream) {
  if (rows < 0 || cols < 0 || side < 0 || side > 2) return TNX_E_INVALID;
  if (rows == 0 || cols == 0) return TNX_OK;
  if (!src || !dst) return TNX_E_INVALID;
  const int64_t total = rows * cols;
  if (rows > 0x7fffffff || cols > 0x7fffffff || (total + 255) / 256 > 0x7fffffffll) return TNX_E_UNSUPPORTED;
  hipLaunchKernelGGL(split_f32_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, src, rows, cols,
                     stride_r, stride_c, (uint16_t*)dst, side);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) { g_last_hip_error = (int)err; return TNX_E_HIP; }
  return TNX_OK;
}

extern "C" int tnx_tile_coords(int schedule, int id, int tiles_m, int tiles_n, int group_m, int* tile_m, int* tile_n) {
  if (!tile_m || !tile_n || tiles_m <= 0 || tiles_n <= 0 || group_m <= 0 || id < 0 ||
      (int64_t)id >= (int64_t)tiles_m * tiles_n || (int64_t)tiles_m * tiles_n > 0x7fffffffll)
    return TNX_E_INVALID;
  // the same functions the kernels call (gemm_tile.h), compiled for the host
  if (schedule & TNX_SCHED_SUPERBLOCK) {
    superblock_order(id, tiles_m, tiles_n, tile_m, tile_n);
  } else {
    const int logical = xcd_remap(id, tiles_m * tiles_n, 8);
    swizzle2d(logical / tiles_n, logical % tiles_n, tiles_m, tiles_n, group_m, tile_m, tile_n);
  }
  return TNX_OK;
}

extern "C" int tnx_kernel_count(void) {
  int ng = 0, n = 0;
  const KernelGroup* g = tnx_kernel_groups(&ng);
  for (int i = 0; i < ng; ++i)
    for (int j = 0; j < g[i].count; ++j) n += g[i].entries[j].dtype != TNX_F32;    // (those are tnx_gemm_f32's own)
  return n;
}

extern "C" const char* tnx_kernel_name(int idx) {
  static thread_local char buf[96];
  int ng = 0;
  const KernelGroup* g = tnx_kernel_groups(&ng);
  for (int i = 0; i < ng; ++i) {
    if (g[i].count > 0 && g[i].entries[0].dtype == TNX_F32) continue;              // groups hold one type
    if (idx < g[i].count) {
      const KernelEntry& e = g[i].entries[idx];
      const char* dn = e.dtype == TNX_F16 ? "f16" : e.dtype == TNX_BF16 ? "bf16" : "i8";
      snprintf(buf, sizeof(buf), "%s %d %d %d %d %d%s%s", dn, e.bm, e.bn, e.bk, e.nw, e.stages, e.generic ? " generic" : "",
               e.persist ? " persistent" : "");
      if (e.fast_bt) strncat(buf, " bt", sizeof(buf) - strlen(buf) - 1);
      if (e.fast_at) strncat(buf, " at", sizeof(buf) - strlen(buf) - 1);
      return buf;
    }
    idx -= g[i].count;
  }
  return nullptr;
}

extern "C" const char* tnx_strerror(int status) {
  switch (status) {
    case TNX_OK: return "ok";
    case TNX_E_INVALID: return "invalid argument";
    case TNX_E_UNSUPPORTED: return "no kernel is built for this tile / dtype / layout";
    case TNX_E_LDS: return "tile configuration exceeds the per-CU LDS budget";
    case TNX_E_WORKSPACE: return "split-K workspace missing or too small";
    case TNX_E_HIP: return "HIP runtime error";
    case TNX_E_STATIC_LIMIT: return "split-K scratch of this launch exceeds TNX_STATIC_WORKSPACE_BYTES (use tnx_gemm with a workspace)";
    default: return "unknown status";
  }
}

extern "C" int tnx_last_hip_error(void) { return g_last_hip_error; }
extern "C" int tnx_version(void) { return TNX_VERSION; }
