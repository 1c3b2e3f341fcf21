// float32 products: both operands cut into bf16 terms in one pass, then one GEMM launch with a binary32 result.
//
// The terms and what they multiply are those of tnx_split_f32 (x = hi + lo, products hi hi + hi lo + lo hi, a non-finite
// element carried by the first copy of its head alone).  Where this pass writes them follows the operand: an A with k
// along its rows and a B with k along its columns keep k contiguous, [row][hi | hi' | lo]; the others keep their own
// contiguous dimension, [hi ; lo ; hi'] planes of k rows.  So every load and store is a run of the operand's own rows,
// whichever way it is transposed, and the GEMM kernel has a loader for each form.  k is padded to 8 per term and to whole
// K slabs in all, the other dimension to 8, with zeros: the GEMM always runs its aligned path.
//
// Bound by memory: 4 bytes read and 6 written per element.  2048^3: both operands 2 x 11.5 -> 14 us (84 MB, 6 TB/s; before,
// one launch per operand, one element per thread and a 64-bit division each), the whole product 67 -> 59 us, the rest of
// it the GEMM at k' = 6144, 1,100 TFLOP/s.  3072 x 3200 x 2822: 241 -> 162 us, with the 256-wide tiles' binary32 epilogue.
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
  int kp8;                 // k rounded up to 8
  int groups;              // 16-byte chunks (8 elements) per row handled, padding included
  int items;               // (row, chunk) pairs
  int64_t pitch;           // elements per scratch row
  int pad;                 // elements (k along the row) or rows (k planes) of zeros after the three terms
  bool planes;             // rows are k: one plane of kp8 rows per term
  bool tail_second;        // terms in the order hi, lo, hi' (B) instead of hi, hi', lo (A)
  FastDiv div;
};

}  // namespace

__device__ __forceinline__ void split_item(const SplitSide& s, int item) {
  const int o = (int)fd_div((uint32_t)item, s.div), g = item - o * s.groups, j0 = g * 8;
  float v[8];
  const float* src = s.src + (int64_t)o * s.so + (int64_t)j0 * s.si;
  if (s.si == 1 && o < s.outer && j0 + 8 <= s.inner) {
    struct __attribute__((packed, aligned(4))) Run { float v[8]; };
    const Run r = *(const Run*)src;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = r.v[e];
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = o < s.outer && j0 + e < s.inner ? src[(int64_t)e * s.si] : 0.0f;
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
  const int64_t step = s.planes ? (int64_t)s.kp8 * s.pitch : (int64_t)s.kp8;
  uint16_t* dst = s.dst + (int64_t)o * s.pitch + j0;
  i32x4 c[3];
  __builtin_memcpy(&c[0], hi, 16);
  __builtin_memcpy(&c[s.tail_second ? 1 : 2], lo, 16);
  __builtin_memcpy(&c[s.tail_second ? 2 : 1], h2, 16);
#pragma unroll
  for (int t = 0; t < 3; ++t) *(i32x4*)(dst + t * step) = c[t];
  const i32x4 zero = {0, 0, 0, 0};
  if (s.planes ? o == s.kp8 - 1 : g == s.groups - 1) {
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

static int64_t up(int64_t v, int64_t q) { return (v + q - 1) / q * q; }

// The bf16 problem a float32 one becomes (pointers into `scratch`, which may be null for a size query), the two sides
// of the pass that fills it, and the scratch bytes.
static int plan(const tnx_gemm_args* a, void* scratch, tnx_gemm_args* g, SplitSide* sa, SplitSide* sb, int64_t* bytes) {
  if (!a || a->in_dtype != TNX_F32 || a->m < 0 || a->n < 0 || a->k < 0 || a->block_k <= 0) return TNX_E_INVALID;
  if (a->out_dtype != TNX_F32) return TNX_E_UNSUPPORTED;
  if (a->m > 0x7fffffff - 64 || a->n > 0x7fffffff - 64 || a->k > (0x7fffffff - 1024) / 3) return TNX_E_UNSUPPORTED;
  *g = *a;
  g->in_dtype = TNX_BF16;
  bool tile_bt = false, tile_at = false;
  gemm_tile_layouts(g, &tile_bt, &tile_at);
  const bool bt = a->stride_bk == 1 && a->stride_bn != 1 && tile_bt;
  const bool at = !bt && a->stride_am == 1 && a->stride_ak != 1 && a->stride_bk != 1 && tile_at;
  const int64_t kp8 = up(a->k, 8), k3 = up(3 * kp8, a->block_k), mp = up(a->m, 8), np = up(a->n, 8);
  const int64_t a_bytes = up((at ? k3 * mp : a->m * k3) * 2, 256), b_bytes = up((bt ? a->n * k3 : k3 * np) * 2, 256);
  *bytes = a_bytes + b_bytes;
  g->k = k3;
  g->a = scratch;
  g->b = (uint8_t*)scratch + a_bytes;
  g->stride_am = at ? 1 : k3; g->stride_ak = at ? mp : 1;
  g->stride_bk = bt ? 1 : np; g->stride_bn = bt ? k3 : 1;
  auto side = [&](SplitSide* s, const void* src, bool planes, int64_t rows, int64_t cols, int64_t so, int64_t si, void* dst,
                  int64_t pitch, bool tail_second) {
    s->src = (const float*)src; s->dst = (uint16_t*)dst;
    s->so = so; s->si = si;
    s->outer = (int)rows; s->inner = (int)cols;
    s->kp8 = (int)kp8;
    s->planes = planes; s->tail_second = tail_second;
    s->pitch = pitch;
    s->pad = (int)(k3 - 3 * kp8);
    const int64_t groups = planes ? pitch / 8 : kp8 / 8, items = (planes ? kp8 : rows) * groups;
    s->groups = (int)groups; s->items = items > 0x7fffffff - 256 ? -1 : (int)items;
    s->div = make_fastdiv((uint32_t)(groups > 0 ? groups : 1));
  };
  if (at) side(sa, a->a, true, a->k, a->m, a->stride_ak, a->stride_am, scratch, mp, false);
  else side(sa, a->a, false, a->m, a->k, a->stride_am, a->stride_ak, scratch, k3, false);
  if (bt) side(sb, a->b, false, a->n, a->k, a->stride_bn, a->stride_bk, (uint8_t*)scratch + a_bytes, k3, true);
  else side(sb, a->b, true, a->k, a->n, a->stride_bk, a->stride_bn, (uint8_t*)scratch + a_bytes, np, true);
  return sa->items < 0 || sb->items < 0 ? TNX_E_UNSUPPORTED : TNX_OK;
}

extern "C" size_t tnx_gemm_f32_scratch_bytes(const tnx_gemm_args* a) {
  tnx_gemm_args g;
  SplitSide sa, sb;
  int64_t bytes = 0;
  return plan(a, nullptr, &g, &sa, &sb, &bytes) == TNX_OK ? (size_t)bytes : 0;
}

extern "C" int tnx_gemm_f32(const tnx_gemm_args* a, void* scratch, size_t scratch_bytes) {
  tnx_gemm_args g;
  SplitSide sa, sb;
  int64_t bytes = 0;
  int st = plan(a, scratch, &g, &sa, &sb, &bytes);
  if (st != TNX_OK) return st;
  if (a->m == 0 || a->n == 0) return TNX_OK;
  if (a->k == 0) {                          // nothing to cut: the GEMM writes zeros
    g.k = 0;
    return tnx_gemm(&g);
  }
  if (!a->a || !a->b || !a->c) return TNX_E_INVALID;
  if (((uintptr_t)a->a | (uintptr_t)a->b | (uintptr_t)a->c) & 3) return TNX_E_INVALID;
  if (!scratch || scratch_bytes < (size_t)bytes || ((uintptr_t)scratch & 255)) return TNX_E_WORKSPACE;
  st = gemm_check(&g, true);                // refuse what the GEMM would refuse before anything is launched
  if (st != TNX_OK) return st;
  const unsigned blocks_a = (unsigned)((sa.items + 255) / 256), blocks_b = (unsigned)((sb.items + 255) / 256);
  hipLaunchKernelGGL(split_f32_pair_kernel, dim3(blocks_a + blocks_b), dim3(256), 0, (hipStream_t)a->stream, sa, sb, blocks_a);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) { note_hip_error((int)err); return TNX_E_HIP; }
  return gemm_launch(&g, nullptr, true);
}
