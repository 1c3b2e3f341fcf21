// float32 products: both operands cut into bf16 terms in one pass, then one GEMM launch with a binary32 result.
//
// x = hi + lo in bf16, products hi hi + lo hi + hi lo in one binary32 sum.  The tiles of the built-in choice take the
// operands once as heads and once as tails, in blocks of 32 k, and form the three products from them (PAIR in
// gemm_tile.h); every other tile gets three copies of k, [hi | hi' | lo] against [hi | lo | hi'], as tnx_split_f32 lays
// them out.  A non-finite element must not meet a tail that happens to be zero (inf * 0): in the three copies it is carried
// by the first head alone; in the pairs its head is +-1 and its tail the element itself, so that against a finite or a
// non-finite partner every product that is not finite has the right sign, and the finite ones vanish beside it.  (Either
// way a partner of at most 2^-134 has a zero head, and an infinity times it gives NaN where float32 gives the infinity.)
// Where this pass writes follows the operand: an A with k along its rows and a B with k along its columns keep k
// contiguous; the others keep their own contiguous dimension, k rows of it.  So every load and store is a run of the
// operand's own rows, whichever way it is transposed, and the GEMM kernel has a loader for each form.  k is padded to
// whole K slabs (pairs: to 32, three copies: to 8 per term), the other dimension to 8, with zeros: the GEMM always runs
// its aligned path.
//
// Bound by memory: 4 bytes read and 4 (three copies: 6) written per element.  2048^3: 13 us for both operands (64 MB, 5 TB/s),
// the product from 61.3 us (three copies) to 52.4; its GEMM, 64 slabs of 0.64 us, is bound by filling the slabs from the L2
// and by the MFMAs (0.45 us of a slab).  3072 x 3200 x 2822: 162 -> 145 us.
//
// Small products and few rows skip all that: the binary32 matrix instruction on the operands as they are (TagF32 in
// gemm_tile.h, chosen by tnx_gemm_f32_config), one launch, no scratch.
#include <hip/hip_runtime.h>
#include <string.h>

#include "../../include/tritonix_hip.h"
#include "registry.h"

using namespace tnx;

namespace {

struct SplitSide {
  const float* src;
  uint16_t* dst;
  int64_t so, si;          // element strides of the source: from row to row of the scratch form, along a row
  int outer, inner;        // rows and columns of the source in that form
  int kp;                  // k rounded up to 8 (pairs: to 32)
  int groups;              // 16-byte chunks (8 elements) per row handled, padding included
  int row0, items;         // first row of this launch, and its (row, chunk) pairs
  int64_t pitch;           // elements per scratch row
  int pad;                 // elements (k along the row) or rows (k planes) of zeros after the three terms
  bool planes;             // rows are k: one plane of kp8 rows per term
  bool tail_second;        // terms in the order hi, lo, hi' (B) instead of hi, hi', lo (A)
  bool pair;               // heads and tails in blocks of 32 k instead of three copies of k
  FastDiv div;
};

}  // namespace

__device__ __forceinline__ void split_item(const SplitSide& s, int item) {
  const int q = (int)fd_div((uint32_t)item, s.div), g = item - q * s.groups, j0 = g * 8, o = s.row0 + q;
  float v[8];
  const float* src = s.src + (int64_t)o * s.so + (int64_t)j0 * s.si;
  if (s.si == 1 && o < s.outer && s.inner - j0 >= 8) {
    struct __attribute__((packed, aligned(4))) Run { float v[8]; };
    const Run r = *(const Run*)src;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = r.v[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = o < s.outer && e < s.inner - j0 ? src[(int64_t)e * s.si] : 0.0f;
  }
  if (s.pair) {
    uint16_t hi[8], lo[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const __bf16 h = (__bf16)v[e];                       // round to nearest even
      const float rest = v[e] - (float)h;
      const bool fin = __builtin_isfinite(rest) && __builtin_isfinite((float)h);
      // (a finite element that rounds to an infinite head counts as that infinity)
      const __bf16 one = __builtin_signbit(v[e]) ? (__bf16)-1.0f : (__bf16)1.0f;
      hi[e] = __builtin_bit_cast(uint16_t, fin ? h : one);
      lo[e] = __builtin_bit_cast(uint16_t, fin ? (__bf16)rest : h);
    }
    // k block o / 32 (planes) or g / 4 of 64 rows or columns: 32 heads, 32 tails
    uint16_t* dst = s.planes ? s.dst + (int64_t)(o / 32 * 64 + o % 32) * s.pitch + j0 : s.dst + (int64_t)o * s.pitch + g / 4 * 64 + g % 4 * 8;
    i32x4 c[2];
    __builtin_memcpy(&c[0], hi, 16);
    __builtin_memcpy(&c[1], lo, 16);
    *(i32x4*)dst = c[0];
    *(i32x4*)(dst + (s.planes ? 32 * s.pitch : 32)) = c[1];
    return;
  }
  uint16_t hi[8], lo[8], h2[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const __bf16 h = (__bf16)v[e];                       // round to nearest even
    const float rest = v[e] - (float)h;
    const bool fin = __builtin_isfinite(rest) && __builtin_isfinite((float)h);
    hi[e] = __builtin_bit_cast(uint16_t, h);
    lo[e] = fin ? __builtin_bit_cast(uint16_t, (__bf16)rest) : (uint16_t)0;
    h2[e] = fin ? hi[e] : (uint16_t)0;
  }
  const int64_t step = s.planes ? (int64_t)s.kp * s.pitch : (int64_t)s.kp;
  uint16_t* dst = s.dst + (int64_t)o * s.pitch + j0;
  i32x4 c[3];
  __builtin_memcpy(&c[0], hi, 16);
  __builtin_memcpy(&c[s.tail_second ? 1 : 2], lo, 16);
  __builtin_memcpy(&c[s.tail_second ? 2 : 1], h2, 16);
#pragma unroll
  for (int t = 0; t < 3; ++t) *(i32x4*)(dst + t * step) = c[t];
  const i32x4 zero = {0, 0, 0, 0};
  if (s.planes ? o == s.kp - 1 : g == s.groups - 1) {
    uint16_t* z = s.planes ? s.dst + 3 * step + j0 : s.dst + (int64_t)o * s.pitch + 3 * step;
    for (int x = 0; x < s.pad; x += s.planes ? 1 : 8) *(i32x4*)(z + (s.planes ? (int64_t)x * s.pitch : x)) = zero;
  }
}

__global__ __launch_bounds__(256) void split_f32_pair_kernel(SplitSide a, SplitSide b, unsigned blocks_a) {
  if (blockIdx.x < blocks_a) {
    const int item = blockIdx.x * 256 + threadIdx.x;
    if (item < a.items) split_item(a, item);
  } else {
    const int item = (int)(blockIdx.x - blocks_a) * 256 + threadIdx.x;
    if (item < b.items) split_item(b, item);
  }
}

// Pairs of one operand per launch: larger operands (2^30 elements, 4 GB of float32) take several, a millisecond each.  Both
// operands' threads then stay within 32 bits, in the pair's number and in the grid.
static constexpr int64_t MAX_ITEMS = 1ll << 27;

static int64_t up(int64_t v, int64_t q) { return (v + q - 1) / q * q; }

// The bf16 problem a float32 one becomes (pointers into `scratch`, which may be null for a size query), the two sides
// of the pass that fills it, and the scratch bytes.
static int plan(const tnx_gemm_args* a, void* scratch, tnx_gemm_args* g, SplitSide* sa, SplitSide* sb, int64_t* bytes, bool* pair) {
  if (!a || a->in_dtype != TNX_F32 || a->m < 0 || a->n < 0 || a->k < 0 || a->block_k <= 0) return TNX_E_INVALID;
  if (a->out_dtype != TNX_F32) return TNX_E_UNSUPPORTED;
  if (a->m > 0x7fffffff || a->n > 0x7fffffff || a->k > (0x7fffffff - 1024) / 3) return TNX_E_UNSUPPORTED;
  *g = *a;
  g->in_dtype = TNX_BF16;
  bool tile_bt = false, tile_at = false;
  gemm_tile_layouts(g, pair, &tile_bt, &tile_at);
  const bool bt = a->stride_bk == 1 && a->stride_bn != 1 && tile_bt;
  const bool at = !bt && a->stride_am == 1 && a->stride_ak != 1 && a->stride_bk != 1 && tile_at;
  // kp: k per term, padded; kt: all terms
  const int64_t kp = up(a->k, *pair ? 32 : 8), kt = *pair ? 2 * kp : up(3 * kp, a->block_k), mp = up(a->m, 8), np = up(a->n, 8);
  const int64_t a_bytes = up((at ? kt * mp : a->m * kt) * 2, 256), b_bytes = up((bt ? a->n * kt : kt * np) * 2, 256);
  *bytes = a_bytes + b_bytes;
  g->k = kt;
  g->a = scratch;
  g->b = (uint8_t*)scratch + a_bytes;
  g->stride_am = at ? 1 : kt; g->stride_ak = at ? mp : 1;
  g->stride_bk = bt ? 1 : np; g->stride_bn = bt ? kt : 1;
  auto side = [&](SplitSide* s, const void* src, bool planes, int64_t rows, int64_t cols, int64_t so, int64_t si, void* dst,
                  int64_t pitch, bool tail_second) {
    s->src = (const float*)src; s->dst = (uint16_t*)dst;
    s->so = so; s->si = si;
    s->outer = (int)rows; s->inner = (int)cols;
    s->kp = (int)kp;
    s->pair = *pair;
    s->planes = planes; s->tail_second = tail_second;
    s->pitch = pitch;
    s->pad = *pair ? 0 : (int)(kt - 3 * kp);
    const int64_t groups = planes ? pitch / 8 : kp / 8;
    s->groups = (int)groups;
    s->row0 = s->items = 0;
    s->div = make_fastdiv((uint32_t)(groups > 0 ? groups : 1));
  };
  if (at) side(sa, a->a, true, a->k, a->m, a->stride_ak, a->stride_am, scratch, mp, false);
  else side(sa, a->a, false, a->m, a->k, a->stride_am, a->stride_ak, scratch, kt, false);
  if (bt) side(sb, a->b, false, a->n, a->k, a->stride_bn, a->stride_bk, (uint8_t*)scratch + a_bytes, kt, true);
  else side(sb, a->b, true, a->k, a->n, a->stride_bk, a->stride_bn, (uint8_t*)scratch + a_bytes, np, true);
  return TNX_OK;
}

// moves a side to its next launch; false: nothing left (items 0)
static bool next_rows(SplitSide* s) {
  const int64_t rows = s->planes ? s->kp : s->outer, row0 = (int64_t)s->row0 + (s->groups > 0 ? s->items / s->groups : 0);
  const int64_t most = s->groups > 0 ? (MAX_ITEMS > s->groups ? MAX_ITEMS / s->groups : 1) : 0, left = rows - row0;
  s->row0 = (int)row0;
  s->items = (int)((left < most ? left : most) * s->groups);
  return s->items > 0;
}

extern "C" size_t tnx_gemm_f32_scratch_bytes(const tnx_gemm_args* a) {
  // (asked before there are pointers, or with others: no scratch only where none of them would need any)
  if (gemm_f32_direct(a, true)) return 0;
  tnx_gemm_args g;
  SplitSide sa, sb;
  int64_t bytes = 0;
  bool pair = false;
  return plan(a, nullptr, &g, &sa, &sb, &bytes, &pair) == TNX_OK ? (size_t)bytes : 0;
}

extern "C" int tnx_gemm_f32(const tnx_gemm_args* a, void* scratch, size_t scratch_bytes) {
  tnx_gemm_args g;
  SplitSide sa, sb;
  int64_t bytes = 0;
  bool pair = false;
  int st = plan(a, scratch, &g, &sa, &sb, &bytes, &pair);
  if (st != TNX_OK) return st;
  if (a->m == 0 || a->n == 0) return TNX_OK;
  if (gemm_f32_direct(a, false)) {
    if (!a->a || !a->b || !a->c || (((uintptr_t)a->a | (uintptr_t)a->b | (uintptr_t)a->c) & 3)) return TNX_E_INVALID;
    return gemm_launch(a, nullptr, GEMM_F32);
  }
  if (a->k == 0) {                          // nothing to cut: the GEMM writes zeros
    g.k = 0;
    return gemm_launch(&g, nullptr, pair ? GEMM_PAIR : GEMM_PADDED);
  }
  if (!a->a || !a->b || !a->c) return TNX_E_INVALID;
  if (((uintptr_t)a->a | (uintptr_t)a->b | (uintptr_t)a->c) & 3) return TNX_E_INVALID;
  st = gemm_check(&g, pair ? GEMM_PAIR : GEMM_PADDED); // refuse what the GEMM would refuse before anything is launched
  if (st != TNX_OK) return st;
  if (!scratch || scratch_bytes < (size_t)bytes || ((uintptr_t)scratch & 255)) return TNX_E_WORKSPACE;
  for (;;) {
    const bool more_a = next_rows(&sa), more_b = next_rows(&sb);
    if (!more_a && !more_b) break;
    const unsigned blocks_a = (unsigned)((sa.items + 255) / 256), blocks_b = (unsigned)((sb.items + 255) / 256);
    hipLaunchKernelGGL(split_f32_pair_kernel, dim3(blocks_a + blocks_b), dim3(256), 0, (hipStream_t)a->stream, sa, sb, blocks_a);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) { note_hip_error((int)err); return TNX_E_HIP; }
  }
  return gemm_launch(&g, nullptr, pair ? GEMM_PAIR : GEMM_PADDED);
}
