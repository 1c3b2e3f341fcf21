// Tiled GEMM for gfx950 (MI355X): C[m,n] = A[m,k] @ B[k,n], optional split-K
// partials and a fused GLU epilogue.
//
// What it computes follows tritonix/ops/matmul.py:43-108 (matmul_kernel),
// :147-202 (gemm_splitk_kernel) and tritonix/ops/swiglu.py:24-110 (glu_kernel):
// a block_m x block_n output tile per workgroup, a K loop of block_k slabs with
// fp32 (int32 for int8) accumulation, an M/N-masked store.  How it computes it
// is specific to CDNA4:
//   * global -> LDS with the 16-byte direct-to-LDS load (no VGPR staging), a
//     ring of STAGES LDS slabs, one workgroup barrier per K slab;
//   * A fragments with ds_read_b128, B fragments (B is row-major [k,n], MFMA
//     wants k-contiguous lanes) with the transposing ds_read_b64_tr_b16/_b8;
//   * XOR-swizzled 16-byte chunks so neither the DMA writes nor the fragment
//     reads collide on LDS banks;
//   * v_mfma_f32_16x16x32 (bf16/f16) and v_mfma_i32_16x16x64_i8 (the 32x32 shapes
//     stay selectable through TileCfg::MI);
//   * a 1-D grid whose block index is remapped XCD-first, then by the
//     group-M order of tl.swizzle2d (tritonix/ops/matmul.py:70).
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include <stdint.h>

// Attribution builds (never the shipped library): -D TNX_LADDER=n strips the K loop of the DMA kernels down to a rung
// of the ladder  1: MFMAs only (both fragment sets filled once from the first slab)  2: + the fragment reads from
// LDS and the per-slab barrier, no refill of the ring  3: + the refill, but always of the tile's first slabs, so every
// load is served by the L2  4: the full loop without its waits for the loads  (0: the kernel as shipped).  Results
// of rungs 1-4 are wrong on purpose; they are timed with power and clock sampling beside the full kernel to say
// what each part of the loop costs on a power-limited board.
#ifndef TNX_LADDER
#define TNX_LADDER 0
#endif
// Development schedule (never the shipped library): -D TNX_PINGPONG=1 runs the K loop of the eight-wave two-slot
// tiles with two k steps per slab as a ping-pong: the two waves of every SIMD alternate, a barrier apart, between
// reading a whole slab's fragments from LDS and multiplying them at raised priority (see pingpong_loop).  Values
// above 1 are its attribution forms: 2 priority not raised; 3 without the fragment reads, 4 without the DMA refill,
// 5 without the MFMAs (3-5: wrong results on purpose).  Measured, it loses to the interleaved loop on every operand.
#ifndef TNX_PINGPONG
#define TNX_PINGPONG 0
#endif

namespace tnx {

typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

#define TNX_LDS(T, addr) ((T __attribute__((address_space(3)))*)(uintptr_t)(addr))

enum { DT_F16 = 0, DT_BF16 = 1, DT_I8 = 2, DT_I32 = 3, DT_F32 = 4 };
enum { EPI_NONE = 0, EPI_GLU_SILU = 1, EPI_GLU_SIGMOID = 2, EPI_GLU_IDENTITY = 3 };

// n / d for 0 <= n < 2^31 by multiply-high and shift (d >= 1); built on the host.
struct FastDiv {
  uint32_t mul, shift;
};
inline FastDiv make_fastdiv(uint32_t d) {
  FastDiv f = {0u, 0u};
  if (d <= 1) return f;
  uint32_t s = 0;
  while ((1ull << s) < d) ++s;
  f.shift = s;
  f.mul = (uint32_t)(((1ull << 32) * ((1ull << s) - d)) / d + 1);
  return f;
}
// the same from its multiplier: the shift follows from the divisor
__device__ __forceinline__ FastDiv fd_of(uint32_t mul, uint32_t d) {
  return FastDiv{mul, d <= 1 ? 0u : 32u - (uint32_t)__builtin_clz(d - 1)};
}
__host__ __device__ __forceinline__ uint32_t fd_div(uint32_t n, FastDiv f) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (__umulhi(n, f.mul) + n) >> f.shift;
#else
  return (uint32_t)((((uint64_t)n * f.mul) >> 32) + n) >> f.shift;
#endif
}

// Geometry of a conv2d forward run on the GEMM kernel (gemm_tile_kernel<..., CONV>): A is the KCRS weight as
// [c_out, c_in*R*S], the B operand is generated from the NCHW input by the DMA loader, column n of the product is
// pixel (image, h_out, w) of a pixel index space whose rows are `wp` wide (w_out rounded up to 8, so that a 16-byte
// chunk of 8 pixels never leaves its output row; the pixels w >= w_out of a row are computed and dropped).
struct ConvGeom {
  int h_in, w_in, c_out, h_out, w_out, wp;
  int stride_h, pad_h, pad_w;
  int hw_in, chw_in;               // h_in*w_in, c_in*h_in*w_in
  int n_total;                     // batch * h_out * wp
  uint32_t x_bytes;                // size of the input tensor
  FastDiv div_hwp, div_wp;         // by h_out*wp, by wp
  FastDiv div_rs, div_s;           // by R*S, by S
  int rs, fw, dil_h, dil_w;
  // one K slab (block_k rows) further along k: what is added to a tap's (dw, dh, element offset), the limits at which
  // dw and dh wrap, and what a wrap adds to the element offset
  int step_dw, step_dh, step_koff, lim_w, lim_h, adj_w, adj_h;
  const uint8_t* bias;             // [c_out] or null
  int bias_dtype;
};

// Geometry of a conv2d forward over a packed input (gemm_tile_kernel<..., GATHER>): the input has been copied to
// [image][row][column][channel], channels in groups of eight, with its zero padding written out, and the weight to
// [c_out][filter tap][channel].  The B operand is then k-contiguous: row n of a slab is 128 bytes of pixel n's window,
// found at (offset of the pixel) + (offset of the slab's filter tap and channels), and nothing in the loader depends
// on the stride, the dilation or where the image ends.
struct PackGeom {
  int hw_out, hwp, w_out;          // pixels of an output plane, the same rounded up to 8, width of an output row
  FastDiv div_hwp, div_w;
  uint32_t img_bytes, row_bytes, col_bytes;   // packed input: one image, one output row, one output column further
  int chunks, cpt, fw;             // 16-byte chunks of k that exist, chunks per filter tap, filter width
  int taps;                        // filter height * width
  FastDiv div_cpt, div_fw, div_taps;
  uint32_t tap_row_bytes, tap_col_bytes;      // one filter row, one filter column further
  uint32_t x_bytes;                // size of the packed input (< 2^31)
};

struct GemmParams {
  const uint8_t* a;
  const uint8_t* b;
  uint8_t* c;
  uint8_t* ws;            // split-K workspace: tile counters, then the slices [slice][cut tile][wave][group][lane]
  int64_t m, n, k;
  int64_t sam, sak;       // element strides of A
  int64_t sbk, sbn;       // element strides of B
  int64_t scm, scn;       // element strides of C
  int tiles_m, tiles_n;
  int group_m;
  int split_k;
  int split_tile0;        // tiles [0, split_tile0) in launch order are computed whole; the rest are cut split_k ways
  int ktiles_per_split;   // K slabs handled by one split
  int epilogue;
  int out_dtype;
  bool c_vec_ok;          // C takes 16-byte stores along n (stride_cn == 1, 16-byte aligned rows)
  bool c_row_ok;          // stride_cn == 1: rows of C take 16-byte stores at the element's own alignment
  int64_t m_load, n_load; // DMA kernels: rows of an m-contiguous A and columns of B that may be loaded (>= m, n: operands padded to whole chunks)
  int tail_slab;          // DMA kernels: the last K slab (whole or partial) is left out of the ring and fetched after the K loop (load_tail)
  bool b_once;            // every element of B is read by exactly one workgroup (one tile row): stream it non-temporally
  int tile_order;         // 0: XCD remap + tl.swizzle2d(group_m); 1: 16x16 super-blocks in serpentine order (superblock_order)
  int atomic_reduce;      // split-K: slices are added into one fp32/int32 copy with device-scope atomics instead of being kept apart
  int batch;              // uncut, non-persistent launches of tiles up to 128x128: the grid holds `batch` problems that share A (0 or 1: one problem);
  int64_t b_batch_bytes, c_batch_bytes;   // problem i reads B + i * b_batch_bytes and writes C + i * c_batch_bytes
  FastDiv div_tiles, div_cut;             // by tiles_m * tiles_n and by the number of cut tiles
  FastDiv div_group, div_rows, div_rows_last;   // by group_m * tiles_n, by the rows of a group and by those of the last, shorter one
  ConvGeom cv;            // read by the CONV kernels; cv.bias / cv.bias_dtype also by the plain epilogue (a bias per row of C)
  PackGeom pk;            // read by the GATHER kernels (with cv's output side)
};

// GemmParams as the kernels with the DMA loader and no conv2d get them (expand_params).  Up to 112 bytes of arguments a launch
// takes the host 2.6 us, from 120 on 3.3 to 3.8, and small products wait for the host: with GemmParams itself (480 bytes)
// 64 x 64 x 64 through tritonix.matmul 5.99 us and 3.28 from C, with these 5.55 and 2.58.  So what a workgroup can work out in a few scalar
// instructions is left out: counts of tiles, unit strides, shifts of divisors.
struct PlainParams {
  const uint8_t* a;
  const uint8_t* b;
  uint8_t* c;
  uint8_t* ws;            // launches of several problems, which cut nothing: the bias
  int64_t lda, ldb;       // of A's rows (AT: of its k), of B's k rows (BT: of its n)
  int64_t scm, scn;
  int32_t m, n, k;
  int32_t group_m, split_k, split_tile0, ktiles_per_split;
  uint32_t mul_tiles;     // multipliers of div_tiles or, with a cut, div_cut;
  uint32_t mul_group, mul_rows, mul_rows_last;
  uint32_t flags;
};
static_assert(sizeof(PlainParams) == 112, "a longer argument list costs every launch 0.7 us");
enum : uint32_t {
  PF_EPILOGUE = 7u, PF_OUT_SHIFT = 3, PF_BIAS_SHIFT = 6,                          // three bits each
  PF_C_VEC = 1u << 9, PF_C_ROW = 1u << 10, PF_TAIL = 1u << 11, PF_B_ONCE = 1u << 12, PF_ORDER = 1u << 13, PF_ATOMIC = 1u << 14,
  PF_PADDED = 1u << 15, PF_MANY = 1u << 16
};

// ---------------------------------------------------------------------------
// element tags
// ---------------------------------------------------------------------------
struct TagF16 { static constexpr int ES = 2; static constexpr int ID = DT_F16; typedef float acc_s; };
struct TagBF16 { static constexpr int ES = 2; static constexpr int ID = DT_BF16; typedef float acc_s; };
struct TagI8 { static constexpr int ES = 1; static constexpr int ID = DT_I8; typedef int acc_s; };
// float32 operands as they are, on the binary32 matrix instruction (a sixteenth of bf16's rate)
struct TagF32 { static constexpr int ES = 4; static constexpr int ID = DT_F32; typedef float acc_s; };

template <class T, int MI> struct Mma;
template <> struct Mma<TagBF16, 32> {
  typedef f32x16 acc_t;
  static __device__ __forceinline__ acc_t run(i32x4 a, i32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma<TagBF16, 16> {
  typedef f32x4 acc_t;
  static __device__ __forceinline__ acc_t run(i32x4 a, i32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma<TagF16, 32> {
  typedef f32x16 acc_t;
  static __device__ __forceinline__ acc_t run(i32x4 a, i32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma<TagF16, 16> {
  typedef f32x4 acc_t;
  static __device__ __forceinline__ acc_t run(i32x4 a, i32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
// 16 k: four instructions of four k.  Lane group g holds k = 4 g .. 4 g + 3 of a 16-byte fragment and gives instruction e
// its element e, so the instructions take the k in another order than they lie in, A and B alike.
template <> struct Mma<TagF32, 16> {
  typedef f32x4 acc_t;
  static __device__ __forceinline__ acc_t run(i32x4 a, i32x4 b, acc_t c) {
    const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], c, 0, 0, 0);
    return c;
  }
};
template <> struct Mma<TagI8, 32> {
  typedef i32x16 acc_t;
  static __device__ __forceinline__ acc_t run(i32x4 a, i32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<TagI8, 16> {
  typedef i32x4 acc_t;
  static __device__ __forceinline__ acc_t run(i32x4 a, i32x4 b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  }
};

// Whether the ring of a tail_slab launch stays inside an operand whose k rows have `len` elements at a pitch of
// `pitch` >= len, `rows` of them in the slab that is left out: the last k row in the ring is loaded in whole chunks too,
// and the rows left out have to reach the end of its last chunk.  They do, unless a row is shorter than a chunk (16-bit
// types: up to 3 elements, int8: up to 7).
__host__ __device__ inline bool ring_chunks_inside(int64_t rows, int64_t len, int64_t pitch, int vec) {
  return rows * pitch + len >= (len + vec - 1) / vec * vec;
}

// ---------------------------------------------------------------------------
// tile-id remap.  Workgroups are dealt round-robin to the 8 XCDs (each has its
// own L2), so consecutive *logical* tile ids are first gathered per XCD, then
// ordered group-M-first exactly like tl.swizzle2d on the row-major tile index
// (triton/language/standard.py:80-116, called at tritonix/ops/matmul.py:70).
// ---------------------------------------------------------------------------
__host__ __device__ inline int xcd_remap(int pid, int total, int nxcd) {
  int q = total / nxcd, r = total % nxcd;
  int x = pid % nxcd, idx = pid / nxcd;
  int start = x * q + (x < r ? x : r);
  return start + idx;
}

__host__ __device__ inline void swizzle2d(int i, int j, int size_i, int size_j, int size_g, int* oi, int* oj) {
  int ij = i * size_j + j;
  int size_gj = size_g * size_j;
  int group_id = ij / size_gj;
  int off_i = group_id * size_g;
  int g = size_i - off_i < size_g ? size_i - off_i : size_g;
  int r = ij % size_gj;
  *oi = off_i + r % g;
  *oj = r / g;
}

// The divisors of the tile-id arithmetic, filled in by the launch.  Five divisions by run-time numbers, one after another
// and 30 instructions each, stood before a workgroup's first load (0.1 us of a launch of 64x64 tiles).
inline void set_order_divisors(GemmParams* p) {
  const int64_t tiles = (int64_t)p->tiles_m * p->tiles_n, cut = tiles - p->split_tile0;
  const int last = p->tiles_m % p->group_m;
  p->div_tiles = make_fastdiv((uint32_t)tiles);
  p->div_cut = make_fastdiv((uint32_t)(cut > 0 ? cut : 1));
  // (a group of more tiles than the grid has is the only group: no tile id reaches the divisor)
  const int64_t group = (int64_t)p->group_m * p->tiles_n;
  p->div_group = make_fastdiv((uint32_t)(group < 0x7fffffff ? group : 0x7fffffff));
  p->div_rows = make_fastdiv((uint32_t)p->group_m);
  p->div_rows_last = make_fastdiv((uint32_t)(last ? last : p->group_m));
}
// swizzle2d of tile id `ij` by these divisors (the same map)
__device__ __forceinline__ void swizzle2d(int ij, const GemmParams& p, int* oi, int* oj) {
  const int group_id = (int)fd_div((uint32_t)ij, p.div_group);
  const int off_i = group_id * p.group_m;
  const bool last = p.tiles_m - off_i < p.group_m;
  const int g = last ? p.tiles_m - off_i : p.group_m;
  const int r = ij - group_id * p.group_m * p.tiles_n;
  const int q = (int)fd_div((uint32_t)r, fd_of(last ? p.div_rows_last.mul : p.div_rows.mul, (uint32_t)g));
  *oi = off_i + r - q * g;
  *oj = q;
}

// false: not a launch that PlainParams can describe.  gemm_launch makes none: strides of 1 along a chunk are what its layouts ask for, a
// split excludes problems and bias there, and the one caller with several problems (conv2d's 1x1 layers) has dense operands -- which
// for one input channel on 1x1 planes count as a k-contiguous B.
inline bool plain_params(const GemmParams& p, bool bt, bool at, int es, PlainParams* q) {
  const bool many = p.batch > 1 || p.cv.bias;
  const int es_out = p.out_dtype == DT_F32 || p.out_dtype == DT_I32 ? 4 : 2;
  if (p.m > 0x7fffffff || p.n > 0x7fffffff || p.k > 0x7fffffff) return false;
  if ((at ? p.sam : p.sak) != 1 || (bt ? p.sbk : p.sbn) != 1) return false;
  if (many && p.split_k > 1) return false;
  if (p.batch > 1 && (p.b_batch_bytes != p.k * p.sbk * es || p.c_batch_bytes != p.m * p.scm * es_out)) return false;
  const bool padded = p.m_load != p.m || p.n_load != p.n;
  if (padded && (p.m_load != (p.m + 7) / 8 * 8 || p.n_load != (p.n + 7) / 8 * 8)) return false;
  q->a = p.a; q->b = p.b; q->c = p.c;
  q->ws = many ? (uint8_t*)p.cv.bias : p.ws;
  q->lda = at ? p.sak : p.sam; q->ldb = bt ? p.sbn : p.sbk;
  q->scm = p.scm; q->scn = p.scn;
  q->m = (int32_t)p.m; q->n = (int32_t)p.n; q->k = (int32_t)p.k;
  q->group_m = p.group_m < p.tiles_m ? p.group_m : p.tiles_m;            // a group of more rows than there are: the same order
  q->split_k = p.split_k; q->split_tile0 = p.split_tile0; q->ktiles_per_split = p.ktiles_per_split;
  GemmParams d;
  d.tiles_m = p.tiles_m; d.tiles_n = p.tiles_n; d.group_m = q->group_m; d.split_tile0 = p.split_tile0;
  set_order_divisors(&d);
  q->mul_tiles = p.split_k > 1 ? d.div_cut.mul : d.div_tiles.mul;
  q->mul_group = d.div_group.mul; q->mul_rows = d.div_rows.mul; q->mul_rows_last = d.div_rows_last.mul;
  q->flags = (uint32_t)p.epilogue | (uint32_t)p.out_dtype << PF_OUT_SHIFT | (p.cv.bias ? (uint32_t)p.cv.bias_dtype << PF_BIAS_SHIFT : 0u) |
             (p.c_vec_ok ? PF_C_VEC : 0u) | (p.c_row_ok ? PF_C_ROW : 0u) | (p.tail_slab ? PF_TAIL : 0u) | (p.b_once ? PF_B_ONCE : 0u) |
             (p.tile_order ? PF_ORDER : 0u) | (p.atomic_reduce ? PF_ATOMIC : 0u) | (padded ? PF_PADDED : 0u) | (many ? PF_MANY : 0u);
  return true;
}
template <class C, bool BT, bool AT> __device__ __forceinline__ GemmParams expand_params(const PlainParams& q) {
  GemmParams p;
  const bool many = (q.flags & PF_MANY) != 0, padded = (q.flags & PF_PADDED) != 0;
  p.a = q.a; p.b = q.b; p.c = q.c; p.ws = q.ws;
  p.m = q.m; p.n = q.n; p.k = q.k;
  p.sam = AT ? 1 : q.lda; p.sak = AT ? q.lda : 1;
  p.sbk = BT ? 1 : q.ldb; p.sbn = BT ? q.ldb : 1;
  p.scm = q.scm; p.scn = q.scn;
  p.tiles_m = (int)(((uint32_t)q.m + C::BM - 1) / C::BM); p.tiles_n = (int)(((uint32_t)q.n + C::BN - 1) / C::BN);
  p.group_m = q.group_m; p.split_k = q.split_k; p.split_tile0 = q.split_tile0; p.ktiles_per_split = q.ktiles_per_split;
  p.epilogue = (int)(q.flags & PF_EPILOGUE); p.out_dtype = (int)(q.flags >> PF_OUT_SHIFT & 7u);
  p.c_vec_ok = (q.flags & PF_C_VEC) != 0; p.c_row_ok = (q.flags & PF_C_ROW) != 0;
  p.tail_slab = (q.flags & PF_TAIL) != 0; p.b_once = (q.flags & PF_B_ONCE) != 0;
  p.tile_order = (q.flags & PF_ORDER) != 0; p.atomic_reduce = (q.flags & PF_ATOMIC) != 0;
  p.m_load = padded ? (p.m + 7) / 8 * 8 : p.m; p.n_load = padded ? (p.n + 7) / 8 * 8 : p.n;
  p.batch = many ? 2 : 1;                                               // one problem or several: what the kernel asks
  p.b_batch_bytes = p.k * p.sbk * C::ES; p.c_batch_bytes = p.m * p.scm * (p.out_dtype == DT_F32 || p.out_dtype == DT_I32 ? 4 : 2);
  const uint32_t tiles = (uint32_t)(p.tiles_m * p.tiles_n);
  p.div_tiles = fd_of(q.mul_tiles, tiles); p.div_cut = fd_of(q.mul_tiles, tiles - (uint32_t)q.split_tile0);
  p.div_group = fd_of(q.mul_group, (uint32_t)(q.group_m * p.tiles_n));
  p.div_rows.mul = q.mul_rows; p.div_rows_last.mul = q.mul_rows_last;
  p.cv.bias = many ? q.ws : nullptr; p.cv.bias_dtype = (int)(q.flags >> PF_BIAS_SHIFT & 7u);
  return p;
}
// One launch of a kernel with one argument, straight from its address: without the stub that <<< >>> calls, 2.6 us instead of 2.75.
inline hipError_t launch_kernel(const void* kernel, unsigned grid, unsigned threads, unsigned lds, hipStream_t stream, void* arg) {
  void* args[] = {arg};
  const hipError_t err = hipLaunchKernel(kernel, dim3(grid), dim3(threads), args, lds, stream);
  if (err != hipSuccess) (void)hipGetLastError();
  return err;
}

template <bool PLAIN> struct KernelParams { typedef GemmParams type; };
template <> struct KernelParams<true> { typedef PlainParams type; };

// Chip-level tile order for grids much larger than the CU count.  The 256 workgroups that run
// together (one per CU) take one 16x16 super-block of tiles, so one "round" touches 16 row panels
// of A and 16 column panels of B; super-blocks are walked in serpentine order, so consecutive
// rounds share half of their operands (which then come from the 256 MiB memory-side cache instead
// of HBM); inside a super-block each XCD owns an 8x4 sub-block (12 panels through its L2).
// A bijection from [0, tiles_m*tiles_n) onto the tile grid for every grid size.
__host__ __device__ inline void superblock_order(int pid, int tiles_m, int tiles_n, int* pm, int* pn) {
  constexpr int SB = 16, CHUNK = SB * SB;
  const int total = tiles_m * tiles_n;
  // ids congruent mod 8 (one XCD) become one run inside each aligned chunk of 256 ids
  const int chunk0 = pid - pid % CHUNK;
  const int csize = total - chunk0 < CHUNK ? total - chunk0 : CHUNK;
  const int s = chunk0 + xcd_remap(pid - chunk0, csize, 8);
  // s-th tile of the walk: rows of super-blocks top to bottom, alternating direction
  const int row_tiles = SB * tiles_n;
  const int i = s / row_tiles;
  int rem = s - i * row_tiles;
  const int h = tiles_m - i * SB < SB ? tiles_m - i * SB : SB;
  const int nsb = (tiles_n + SB - 1) / SB;
  const int wlast = tiles_n - (nsb - 1) * SB;
  const bool rev = i & 1;
  int jw, w;
  if (!rev) {
    jw = rem / (h * SB);
    if (jw > nsb - 1) jw = nsb - 1;
    w = jw == nsb - 1 ? wlast : SB;
    rem -= jw * h * SB;
  } else if (rem < h * wlast) {
    jw = 0;
    w = wlast;
  } else {
    rem -= h * wlast;
    jw = 1 + rem / (h * SB);
    w = SB;
    rem -= (jw - 1) * h * SB;
  }
  const int j = rev ? nsb - 1 - jw : jw;
  int r, c;
  if (h == SB && w == SB) {
    const int sub = rem / 32, idx = rem % 32;     // XCD sub-block: 2 x 4 of them, each 8 rows x 4 columns, walked down the rows
    r = 8 * (sub / 4) + idx % 8;
    c = 4 * (sub % 4) + idx / 8;
  } else {
    r = rem % h;
    c = rem / h;
  }
  *pm = i * SB + r;
  *pn = j * SB + c;
}

// vmcnt-only wait (lgkmcnt and expcnt left at "no wait") in the gfx9 encoding
#define TNX_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | ((((n) >> 4) & 0x3) << 14) | 0x0F70)

// 16 bytes per lane, global -> LDS without touching VGPRs.  LDS destination is
// lds_base + lane*16 (lds_base wave-uniform, carried in M0).  M0 is written inside the asm and
// cannot be named as clobbered (the compiler reserves it and rejects it in a clobber list); that
// is sound only while no compiler-generated instruction of these kernels reads M0 -- none does
// (no register-indexed arrays, no LDS-direct or GWS operations: every array is fully unrolled).
// The builtin form of this load is not used because the compiler then waits for vmcnt(0) before
// every later LDS read, which serialises the ring.
__device__ __forceinline__ void dma16(const uint8_t* sbase, uint32_t voff, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_base), "v"(voff), "s"(sbase)
               : "memory");
}

// The same load in two parts, so that a useful instruction (an LDS read) can take the place of the wait
// state the hardware needs between the write of M0 and the load that uses it.  Nothing that reads or
// writes M0 may be placed between the two.
__device__ __forceinline__ void dma16_set_m0(uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0" : : "s"(lds_base) : "memory");
}
template <bool NT> __device__ __forceinline__ void dma16_go(const uint8_t* sbase, uint32_t voff) {
  if (NT) asm volatile("global_load_lds_dwordx4 %0, %1 nt" : : "v"(voff), "s"(sbase) : "memory");
  else asm volatile("global_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase) : "memory");
}

// same, with the non-temporal hint: for an operand that is streamed from HBM once and never reused
__device__ __forceinline__ void dma16_nt(const uint8_t* sbase, uint32_t voff, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
               :
               : "s"(lds_base), "v"(voff), "s"(sbase)
               : "memory");
}

__device__ __forceinline__ const uint8_t* uniform_ptr(const uint8_t* p) {
  uint64_t v = (uint64_t)(uintptr_t)p;
  uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const uint8_t*)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

// Device-scope (all XCDs) 16-byte accesses for data that workgroups hand to each other inside one kernel,
// as raw buffer operations with the sc1 bit: on gfx942/gfx950 that is the encoding of a monotonic atomic
// access at agent scope (the store writes through the XCD's L2, the load does not hit a stale line of it),
// so no whole-cache write-back or invalidate is needed around them.  They are compiler builtins, so the
// compiler itself places the s_waitcnt before the first use of a loaded value.
constexpr int CPOL_SC1 = 16;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t agent_window(const void* base) {
  // raw buffer (stride 0) of 4 GiB - 1 bytes starting at base; offsets are unsigned 32-bit
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0xffffffff, 0x00020000);
}
__device__ __forceinline__ void store16_agent(__amdgpu_buffer_rsrc_t w, uint32_t off, i32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(v, w, off, 0, CPOL_SC1);
}
__device__ __forceinline__ i32x4 load16_agent(__amdgpu_buffer_rsrc_t w, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(w, off, 0, CPOL_SC1);
}

// 16 bytes of C, stored with the non-temporal hint.  C is written once and never read by the kernel; without the
// hint its lines are kept in the L2 and the memory-side cache and push out operand panels that the other tiles of the
// round still need.  Measured on the 8192^3 bf16 problem: 1531 -> 1595 TFLOP/s on data-like operands (power-limited),
// 1712 -> 2026 on all-zero operands (clock at its maximum: the memory side decides); the gated GEMM 1414 -> 1475,
// int8 2798 -> 2845 TOP/s.  (The same hint on the B *loads* costs 4-20 %: operands are re-read.)
// A launch whose output the next launch reads at once (the feed-forward block's up-projection) loses that read's
// cache hits: the block's down-projection runs ~22 us slower, less than the ~30 us its up-projection gains.
// (A run-time switch `if (keep) plain store else hinted store` is no way to have both: the compiler sinks the two
// stores into one and drops the hint, measured as the full loss of the gain.)
typedef i32x4 __attribute__((aligned(2))) i32x4_loose;
typedef i32x4 __attribute__((aligned(1))) i32x4_bytes;
typedef i32x4 __attribute__((aligned(4))) i32x4_words;
__device__ __forceinline__ void store16_stream(void* dst, i32x4 v) { __builtin_nontemporal_store(v, (i32x4*)dst); }
__device__ __forceinline__ void store16_stream_loose(void* dst, i32x4 v) { __builtin_nontemporal_store(v, (i32x4_loose*)dst); }

// half a fragment from a slab of k rows, ROWB bytes each: 8 bytes along k per lane.  Transposing reads for 16-bit and int8
// elements, two words for 32-bit ones.
template <int ES, int ROWB> __device__ __forceinline__ i32x2 lds_read_tr(uint32_t addr) {
  if constexpr (ES == 2) return __builtin_bit_cast(i32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(TNX_LDS(i16x4, addr)));
  else if constexpr (ES == 1) return __builtin_amdgcn_ds_read_tr8_b64_v2i32(TNX_LDS(i32x2, addr));
  else return i32x2{*TNX_LDS(int, addr), *TNX_LDS(int, addr + ROWB)};
}

__device__ __forceinline__ float quad_swap1(float v) {
  // lanes (0,1,2,3) <- (1,0,3,2)
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}

// 1 / d for d >= 1, as the division rounds it and at two thirds of its instructions: what a general one does for its range and for
// a correction of the quotient falls away.  One Newton step with exact remainders takes the reciprocal instruction's last bit
// (wrong for a ninth of all d) to the correct one.  Past 2^96 the argument is scaled, since that instruction flushes subnormal
// results; at infinity the remainder is no number, and the bound on it leaves 0.  Compared with 1.0f / d on all 1.1e9 d: equal but for
// five subnormal results, which are one unit of 2^-149 off.
__device__ __forceinline__ float reciprocal_from_one(float d) {
  const float c = d > 0x1p96f ? 0x1p-32f : 1.0f;
  const float r = __builtin_amdgcn_rcpf(d * c) * c;
  const float e = __builtin_fmaxf(__builtin_fmaf(-d, r, 1.0f), -1.0f);
  return __builtin_fmaf(e, r, r);
}

// ROUNDED: to 16 bits.  4096 x 28672, gated, bf16: k = 4096 674 us, with the division 671, with the bare instruction 668; k = 512
// 122.2, 129.5 and 118.9; 1024 x 4096 x 64 5.15, 5.27 and 5.02 us.
template <bool ROUNDED> __device__ __forceinline__ float glu_gate(float g, int epi) {
  if (epi == EPI_GLU_IDENTITY) return g;
  const float d = 1.0f + __expf(-g);
  const float s = ROUNDED ? reciprocal_from_one(d) : 1.0f / d;
  return epi == EPI_GLU_SILU ? g * s : s;
}

__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);  // quiet NaN
  u += 0x7fffu + ((u >> 16) & 1u);                                             // round to nearest even
  return (uint16_t)(u >> 16);
}

template <class ACC> __device__ __forceinline__ void store_out(uint8_t* c, int64_t off, ACC v, int out_dtype);
template <> __device__ __forceinline__ void store_out<float>(uint8_t* c, int64_t off, float v, int out_dtype) {
  if (out_dtype == DT_BF16) ((uint16_t*)c)[off] = f32_to_bf16(v);
  else if (out_dtype == DT_F16) ((_Float16*)c)[off] = (_Float16)v;
  else ((float*)c)[off] = v;
}
template <> __device__ __forceinline__ void store_out<int>(uint8_t* c, int64_t off, int v, int out_dtype) {
  ((int*)c)[off] = v;
}

// ---------------------------------------------------------------------------
// static description of one tile configuration
// ---------------------------------------------------------------------------
template <class T, int BM_, int BN_, int BK_, int NW_, int STAGES_>
struct TileCfg {
  static constexpr int ES = T::ES;
  static constexpr int BM = BM_, BN = BN_, BK = BK_, NW = NW_, STAGES = STAGES_;
  static constexpr int THREADS = NW * 64;
  static constexpr int WGM = (NW == 4) ? 2 : (BM > BN ? 4 : 2);  // wave grid
  static constexpr int WGN = NW / WGM;
  static constexpr int WTM = BM / WGM, WTN = BN / WGN;            // wave tile
  // MFMA shape: 16x16 (x32 for 16-bit, x64 for int8).  With operands that toggle like real data the part runs
  // against its board-power limit, and per multiply-add the 16x16 instructions draw measurably less than the
  // 32x32 ones (an MFMA-only loop on random registers sustains 11-15 % more with them, for all three types),
  // which outweighs their four points of extra issue overhead.  The 32x32 code paths below stay usable
  // (MI = 32 needs WTM % 32 == 0 && WTN % 32 == 0).
  static constexpr int MI = 16;
  static_assert(ES != 4 || MI == 16, "binary32 operands: 16x16 shapes only");
  static constexpr int TM = WTM / MI, TN = WTN / MI;
  static constexpr int KB = (MI == 32) ? 32 : 64;                 // k bytes one MFMA consumes
  static constexpr int MMA_K = KB / ES;
  static constexpr int KSTEPS = (BK * ES) / KB;
  static constexpr int KGROUPS = 64 / MI;                         // lane groups along k
  static constexpr int ROWB_A = BK * ES, CPR_A = ROWB_A / 16;
  static constexpr int ROWB_B = BN * ES, CPR_B = ROWB_B / 16;
  static constexpr int A_BYTES = BM * ROWB_A, B_BYTES = BK * ROWB_B;
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int LDS_BYTES = STAGES * STAGE_BYTES;
  static constexpr int A_LOADS = A_BYTES / 1024, B_LOADS = B_BYTES / 1024;  // wave-wide 1 KiB DMA ops
  static constexpr int A_LPW = (A_LOADS + NW - 1) / NW, B_LPW = (B_LOADS + NW - 1) / NW;
  static constexpr int LPW = A_LPW + B_LPW;                       // DMA ops one wave issues per slab
  static constexpr int ACC_N = (MI == 32) ? 16 : 4;
  static constexpr bool VALID_ANY =
      (WTM % 16 == 0) && (WTN % 16 == 0) && (BK * ES) % KB == 0 && KSTEPS >= 1 && CPR_A >= 4 && A_BYTES % 1024 == 0 &&
      B_BYTES % 1024 == 0 && A_LOADS % NW == 0 && LDS_BYTES <= 163840 && TM * TN * ACC_N <= 256 && (STAGES - 2) * LPW <= 63 && STAGES >= 2;
  static constexpr bool VALID = VALID_ANY && CPR_B >= 8 && CPR_B % (ES == 1 ? 4 : 8) == 0 && B_LOADS % NW == 0;
  // GATHER: the B slab has the layout of the A slab, so its width only has to be whole DMA ops (8 rows); ops that do
  // not divide over the waves are issued twice (the same bytes to the same place)
  // AT: the A slab is BK rows of BM elements, read like a row-major B slab
  static constexpr bool VALID_AT = VALID && BM * ES / 16 >= 8 && (BM * ES / 16) % (ES == 1 ? 4 : 8) == 0 && KSTEPS % 2 == 0;
  static constexpr bool VALID_GATHER = VALID_ANY && ES == 2 && BK * ES == 128 && BN % 16 == 0;

  // chunk-index XOR applied to row `row` of the A slab.  A fragment read is one ds_read_b128 with lane = 16 * kg +
  // row: the LDS serves it in four cycles of 16 lanes, and the 16 are not consecutive lanes -- measured with a
  // one-wave probe and SQ_LDS_BANK_CONFLICT, lanes {0-3, 12-15, 20-27} share a cycle and {4-11, 16-19, 28-31} the
  // next (the same again from lane 32), i.e. all 16 rows of the fragment, but rows 4-11 with the neighbouring k
  // chunk.  The XOR therefore has to place rows r, r + 4, r + 8, r + 12 (which share the banks of a 128- or 64-byte
  // row) so that chunk kg of two of them and chunk kg ^ 1 of the other two fall on four different slots; both
  // formulas below do, and the probe counts no conflict cycle for them (the previous pair, (row & 7) ^ (row >> 3 & 1)
  // and (row >> 1 & 3) ^ (row >> 3 & 1), assumed 16 consecutive lanes per cycle and took 8 cycles per read, not 4).
  static __host__ __device__ constexpr int swzA(int row) {
    return CPR_A >= 8 ? ((row & 7) ^ ((row >> 2) & 1)) : (((row >> 3) & 1) << 1);
  }
  // chunk-index XOR applied to row `row` (a k index) of the B slab
  // (A transposing read serves the four 16-lane groups of a wave in two passes; with 16x16 MFMA tiles the two
  // groups of a pass read the same columns 8 k rows apart (16 for int8), so one more row bit enters the XOR to
  // keep them on different banks: it moves the second group onto exactly the chunk slots the first leaves free.)
  static __host__ __device__ constexpr int swzB(int row) { return swzT<CPR_B>(row); }
  // the same for any slab of k rows that transposing reads serve, CPR chunks per row
  template <int CPR> static __host__ __device__ constexpr int swzT(int row) {
    if (ES == 2) {
      const int pass = MI == 16 ? (((row >> 3) ^ (row >> 4)) & 1) << 1 : 0;
      if (CPR % 16 == 0) { int k = row & 3; return ((2 * k + (k >> 1)) << 1) ^ pass; }
      return ((row & 3) << 1) ^ pass;       // stays inside a group of 8 chunks: also for rows of 24 chunks (BN = 192)
    } else if (ES == 4) {
      // a read is 16 neighbouring words (4 chunks) of one k row per lane group, the groups 4 rows apart
      return ((row >> 2) & (CPR % 16 == 0 ? 3 : 1)) << 2;
    } else {
      const int pass = MI == 16 ? ((row >> 4) ^ (row >> 5)) & 1 : 0;
      if (CPR % 16 == 0) { int k = row & 7; return (2 * k + (k >> 2)) ^ pass; }
      if (CPR % 8 == 0) return (row & 7) ^ pass;
      // Rows of 12 chunks (BN = 192), 192 bytes: consecutive rows already start 48 banks apart, so the 8 rows of a
      // 16-lane group only collide with the row 4 below, and the two groups of a pass (rows r and r + 16) with each
      // other: one XOR bit for each, inside a group of 4 chunks.
      return ((row >> 2) & 1) | (((row >> 4) & 1) << 1);
    }
  }
};

template <class X> struct TypeTag { typedef X type; };
template <bool B> struct BoolTag { static constexpr bool value = B; };
template <int V> struct IntTag { static constexpr int value = V; };

// ---------------------------------------------------------------------------
// output conversion and the store of a wave's accumulators
// ---------------------------------------------------------------------------
struct OutBF16 {
  typedef uint16_t raw;
  static __device__ __forceinline__ raw cvt(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }  // RNE
};
struct OutF16 {
  typedef uint16_t raw;
  static __device__ __forceinline__ raw cvt(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
};
// binary32 output of a 16-bit-float GEMM: the accumulator as it is.  It is what lets a float32 product run on the
// bf16 matrix instructions as a three-term split (each operand is cut into a bf16 head and a bf16 tail); built for the
// tiles up to 128x128 (f32_out_tile), for the head-and-tail kernels of any width (PAIR) and for conv2d's.
struct OutF32 {
  typedef float raw;
  static __device__ __forceinline__ raw cvt(float v) { return v; }
};
template <class T> struct OutOf;
template <> struct OutOf<TagBF16> { typedef OutBF16 type; };
template <> struct OutOf<TagF16> { typedef OutF16 type; };
template <> struct OutOf<TagI8> { typedef int type; };
template <> struct OutOf<TagF32> { typedef OutF32 type; };


// LDS one wave needs to pass one row-block (MI rows) of its outputs through LDS: up to 32 bits per accumulator, rows
// padded by 16 bytes to spread the banks.
template <class C> struct EpiStage {
  static constexpr int PITCH = C::WTN * 4 + 16;
  static constexpr int ROWS = C::MI;
  static constexpr int WAVE_BYTES = ROWS * PITCH;
  static constexpr int BYTES = C::NW * WAVE_BYTES;
};

// Outputs of four accumulators of one row (four consecutive columns; GLU: two gate / linear pairs), as they go to the strip.
template <class O, class S, bool GLU> struct Quad;
template <class O, bool GLU> struct Quad<O, float, GLU> {
  typedef typename O::raw raw;
  static constexpr int N = GLU ? 2 : 4;
  typedef raw vec __attribute__((ext_vector_type(N)));
  static __device__ __forceinline__ vec run(float a, float b, float c, float d, int epi) {
    constexpr bool ROUNDED = sizeof(raw) == 2;
    if constexpr (GLU) return vec{O::cvt(glu_gate<ROUNDED>(a, epi) * b), O::cvt(glu_gate<ROUNDED>(c, epi) * d)};
    else return vec{O::cvt(a), O::cvt(b), O::cvt(c), O::cvt(d)};
  }
};
template <bool GLU> struct Quad<int, int, GLU> {
  typedef int raw;
  static constexpr int N = 4;
  typedef int vec __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ vec run(int a, int b, int c, int d, int) { return vec{a, b, c, d}; }
};

// 16 bytes of output from NF accumulator values that sit row-major in LDS.
// GLU: values come in (gate, linear) pairs, one output per pair.
template <class O, class S, bool GLU> struct Pack16;
template <class O, bool GLU> struct Pack16<O, float, GLU> {   // 16-bit float outputs: 8 per lane
  typedef typename O::raw raw;
  static constexpr int OUTV = 8, NF = GLU ? 16 : 8;
  static __device__ __forceinline__ void run(const float* f, int epi, raw* out) {
#pragma unroll
    for (int x = 0; x < OUTV; ++x) out[x] = O::cvt(GLU ? glu_gate<true>(f[2 * x], epi) * f[2 * x + 1] : f[x]);
  }
};
template <bool GLU> struct Pack16<OutF32, float, GLU> {       // binary32 outputs: 4 per lane
  typedef float raw;
  static constexpr int OUTV = 4, NF = GLU ? 8 : 4;
  static __device__ __forceinline__ void run(const float* f, int epi, raw* out) {
#pragma unroll
    for (int x = 0; x < OUTV; ++x) out[x] = GLU ? glu_gate<false>(f[2 * x], epi) * f[2 * x + 1] : f[x];
  }
};
template <bool GLU> struct Pack16<int, int, GLU> {            // int32 outputs: 4 per lane
  typedef int raw;
  static constexpr int OUTV = 4, NF = 4;
  static __device__ __forceinline__ void run(const int* f, int, raw* out) {
#pragma unroll
    for (int x = 0; x < 4; ++x) out[x] = f[x];
  }
};

// Where the split-K slices of one wave's part of a tile sit in the workspace.  A slice is
// stored exactly as the wave holds it: group q = (i*TN + j)*NGRP + g of four accumulator
// registers is one 16-byte element per lane at q*1024 + lane*16, so every store and load
// instruction moves one contiguous KiB.
struct SliceSrc {
  const uint8_t* base;     // this wave's part of slice 0
  uint32_t slice_stride;   // bytes from one slice to the next (the host keeps nslices * slice_stride under 4 GiB)
  int nslices;
  bool rezero;             // atomic reduction: the one slice holds the finished sums; it is cleared again after the read
};

// Workgroups of a tile that a CU is to hold at once, as many as the ring's LDS allows, and the registers a lane may then
// use.  Left to itself the compiler takes all that the hand-over of cut tiles can use (its loads in flight), which the
// launches that cut nothing pay for too: 64x128 tiles of 8 waves on 152 registers, one workgroup on a CU instead of two,
// ran conv2d's 1x1 layer of 1088 -> 320 channels on 14x14, batch 32, in 28.5 us; on 110 registers in 20.5.  NEED: accumulators,
// two sets of fragments and what addresses take; a tile that needs more than its share keeps fewer workgroups resident.  (25 of the
// 681 kernels spill, all of them 256x256 tiles, which one workgroup fills whatever is stated here.)
template <class C> struct Residency {
  static constexpr int LDS = C::LDS_BYTES > EpiStage<C>::BYTES ? C::LDS_BYTES : EpiStage<C>::BYTES;
  static constexpr int ACC = C::TM * C::TN * C::ACC_N;
  static constexpr int NEED = ACC + ACC / 8 + (C::TM + C::TN) * 8 + 24;
  static constexpr int regs_of(int wgs) { return 512 / (wgs * C::NW / 4) / 8 * 8; }
  static constexpr int fit() {
    int r = 163840 / LDS;
    if (r * C::NW > 32) r = 32 / C::NW;
    while (r > 1 && regs_of(r) < NEED) --r;
    return r;
  }
  static constexpr int WGS = fit();
  static constexpr int WAVES = WGS * C::NW / 4;         // per SIMD
  static constexpr int REGS = regs_of(WGS);
};

// largest divisor of n that is <= cap
constexpr int slice_batch(int n, int cap) {
  int g = cap < n ? cap : n;
  while (n % g) --g;
  return g;
}

// Sums of the slices of CG groups, from group c0 of the wave's part on, into the accumulators of those groups; ZB slices in flight
// together, in slice order whatever ZB is.
template <class C, int CG, int ZB, class ACC>
__device__ __forceinline__ void collect_groups(ACC (&acc)[C::TM][C::TN], __amdgpu_buffer_rsrc_t win, const SliceSrc& src, int lane, int c0,
                                               int row_blocks) {
  constexpr int NGRP = C::ACC_N / 4, NQ = C::TN * NGRP, G = C::TM * NQ;
  typedef std::remove_reference_t<decltype(acc[0][0][0])> acc_s;
  typedef acc_s acc4 __attribute__((ext_vector_type(4)));
  acc4 v[CG];
#pragma unroll
  for (int x = 0; x < CG; ++x) v[x] = acc4{0, 0, 0, 0};
  if (c0 / NQ < row_blocks) {
#pragma unroll 1
    for (int z0 = 0; z0 < src.nslices; z0 += ZB) {
      i32x4 w[ZB * CG];
#pragma unroll
      for (int u = 0; u < ZB; ++u) {
        if (z0 + u >= src.nslices) break;
#pragma unroll
        for (int x = 0; x < CG; ++x) {
          // (row-block by row-block in the tiles of few groups; a branch more in the others keeps the compiler from
          // having the loads in flight together at all)
          if (G <= 8 && (c0 + x) / NQ >= row_blocks) break;
          w[u * CG + x] = load16_agent(win, (uint32_t)lane * 16u + (uint32_t)(c0 + x) * 1024u + (uint32_t)(z0 + u) * src.slice_stride);
        }
      }
#pragma unroll
      for (int u = 0; u < ZB; ++u) {
        if (z0 + u >= src.nslices) break;
#pragma unroll
        for (int x = 0; x < CG; ++x) {
          acc4 t;
          __builtin_memcpy(&t, &w[u * CG + x], 16);
          v[x] += t;
        }
      }
    }
  }
#pragma unroll
  for (int x = 0; x < CG; ++x)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[(c0 + x) / NQ][(c0 + x) % NQ / NGRP][(c0 + x) % NGRP * 4 + e] = v[x][e];
}

// The split-K slices of one wave's part of a tile, added in slice order into the accumulators (which an uncut tile
// would hold there), whatever workgroup does it.  Bound by the latency of device-scope loads and, from 64 KiB of slices on,
// by the 64 bytes per cycle a CU takes in: ZB slices of CG groups, 16 to 32 loads per lane, are in flight together, across
// row-blocks.  Nothing is loaded past the last slice (a load from an empty window costs as much) nor, in the tiles of few groups,
// past the last row-block.  What is loaded beyond the problem's rows -- the other lanes of a row-block, the other row-blocks of a batch
// of groups -- was never written: it lies inside the slice, stays in the lane of its row, and no epilogue stores it.
// One row-block alone has fewer groups, so more of its slices fit the same registers: 8 x 2048 x 10240 int8, sixteen cuts, 11.5 us with
// four slices of two row-blocks in flight, 10.8 with eight of one.
template <class C, class ACC>
__device__ __forceinline__ void collect_slices(ACC (&acc)[C::TM][C::TN], const SliceSrc& src, int lane, int64_t rows_left) {
  constexpr int NQ = C::TN * (C::ACC_N / 4), G = C::TM * NQ;
  constexpr int CG = slice_batch(G, G >= 32 ? 8 : 16);
  constexpr int ROOM = (Residency<C>::REGS - 32) / (4 * CG) - 1;        // slices of CG groups beside their sums
  constexpr int ZCAP = G > 8 ? 2 : G == 8 ? 4 : 8;
  constexpr int ZB = ROOM >= ZCAP ? ZCAP : ROOM >= 4 ? 4 : ROOM >= 2 ? 2 : 1;
  constexpr int ZB1 = ZB * CG / NQ < 8 ? ZB * CG / NQ : 8;              // of the first row-block alone
  constexpr bool FEW = G <= 8 && C::TM > 1 && CG > NQ && ZB1 > ZB;
  const __amdgpu_buffer_rsrc_t win = agent_window(src.base);
  const int row_blocks = rows_left >= C::WTM ? C::TM : (int)((rows_left + C::MI - 1) / C::MI);
  if (FEW && row_blocks <= 1) {
#pragma unroll
    for (int i = 1; i < C::TM; ++i)
#pragma unroll
      for (int j = 0; j < C::TN; ++j) acc[i][j] = {};
    collect_groups<C, FEW ? NQ : CG, FEW ? ZB1 : ZB>(acc, win, src, lane, 0, row_blocks);
  } else {
#pragma unroll
    for (int c0 = 0; c0 < G; c0 += CG) collect_groups<C, CG, ZB>(acc, win, src, lane, c0, row_blocks);
  }
  if (src.rezero) {
    // atomic reduction: what was just read is the sum; leave zeros behind for the next launch
    TNX_WAIT_VM(0);
#pragma unroll 1
    for (int q = 0; q < G; ++q) store16_agent(win, (uint32_t)lane * 16u + (uint32_t)q * 1024u, i32x4{0, 0, 0, 0});
  }
}

template <class C> constexpr bool multi_problem_tile() { return C::BM * C::BN <= 128 * 128; }
// tiles whose kernels carry a second copy of the epilogue that writes binary32 (16-bit float inputs only)
template <class T, class C> constexpr bool f32_out_tile() { return T::ES == 2 && C::BM * C::BN <= 128 * 128; }

__device__ __forceinline__ float bias_value(const uint8_t* bias, int row, int dtype) {
  if (dtype == DT_F32) return ((const float*)bias)[row];
  if (dtype == DT_F16) return (float)((const _Float16*)bias)[row];
  return __builtin_bit_cast(float, (uint32_t)((const uint16_t*)bias)[row] << 16);
}

// The bias of a lane's row in each of TM row-blocks, for rows_left >= 1 rows (rows past them get the last one's).  All the loads
// are under way before the first value is converted: one memory round trip, where a value at a time took TM of them.
template <int TM, int MI>
__device__ __forceinline__ void bias_of_rows(const uint8_t* bias, int dtype, int row0, int rows_left, int lane, float (&out)[TM]) {
  uint32_t raw[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = i * MI + lane % MI, row = row0 + (r < rows_left ? r : rows_left - 1);
    raw[i] = dtype == DT_F32 ? ((const uint32_t*)bias)[row] : (uint32_t)((const uint16_t*)bias)[row];
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
    out[i] = dtype == DT_F32   ? __builtin_bit_cast(float, raw[i])
             : dtype == DT_F16 ? (float)__builtin_bit_cast(_Float16, (uint16_t)raw[i])
                               : __builtin_bit_cast(float, raw[i] << 16);
}

// How the lanes of a wave share the 16-byte output chunks of one row-block (ROWS rows of CPRW chunks each), 64 chunks per
// pass.  EVEN: a lane's chunk column is the same in every pass and its row RSTEP further on.
template <int ROWS, int CPRW> struct RowPasses {
  static constexpr int ITERS = (ROWS * CPRW + 63) / 64;
  static constexpr bool EVEN = 64 % CPRW == 0;
  static constexpr int RSTEP = EVEN ? 64 / CPRW : 0;
  static constexpr int NL = EVEN ? 1 : ITERS;           // distinct (row, column) places of a lane
  // passes whose LDS reads are in flight together; the rest, if any, in a rolled loop where the places allow it
  static constexpr int UNR = ITERS <= 4 ? ITERS : (ITERS % 4 == 0 ? 4 : ITERS % 3 == 0 ? 3 : ITERS % 2 == 0 ? 2 : 1);
};

// The MFMA result is C^T: lane l owns output row m = l % MI and, per group of four accumulator
// registers, four consecutive columns n.  Each wave passes one row-block at a time through its
// private LDS strip: gated and rounded outputs in (one write per group), then the strip is read
// row-major and stored 16 bytes per lane, so every row of C receives full contiguous runs.
// Bound, on launches of a round or two of tiles, by its own instructions and LDS traffic: so the outputs are rounded before
// the strip (half the bytes, a quarter for a gated pair), a lane's place in C and in the strip is worked out once, a pass
// adds a scalar, and the next row-block is written to the strip behind the reads of the present one, before its stores
// (a wave's LDS operations are carried out in order: no wait is needed between them).  Sums through the strip, rounded
// after it, with every address worked out anew: 4 tiles of 128x256 and 4 K slabs 7.7 us a launch, now 7.1; of 128x128 5.6, now 5.3;
// the gated 4096 x 28672 x 4096 with its division by a reciprocal too (7 rounds) 1.5 % of the feed-forward block.
template <class T, class C, class O, bool GLU, bool BIAS = false, class ACC>
__device__ __forceinline__ void epilogue_store(ACC (&acc)[C::TM][C::TN], uint8_t* cbase, uint32_t lds_strip, int lane,
                                               int64_t gm0, int64_t gc0, int64_t m, int64_t ncols, int64_t scm, int64_t scn,
                                               bool vec_ok, int epi, const uint8_t* bias = nullptr, int bias_dtype = 0) {
  typedef typename T::acc_s acc_s;
  typedef std::conditional_t<std::is_same<acc_s, int>::value, Quad<int, int, GLU>, Quad<O, acc_s, GLU>> QD;
  typedef typename QD::raw raw;
  constexpr int MI = C::MI;
  constexpr int NGRP = C::ACC_N / 4;                    // groups of four consecutive columns per accumulator tile
  constexpr int OUTV = 16 / sizeof(raw);
  constexpr int WCOLS = GLU ? C::WTN / 2 : C::WTN;      // output columns of the wave tile
  constexpr int PITCH = WCOLS * sizeof(raw) + 16;
  constexpr int CPRW = WCOLS / OUTV;                    // 16-byte output chunks per strip row
  typedef RowPasses<MI, CPRW> RP;
  static_assert(WCOLS % OUTV == 0, "wave tile too narrow for 16-byte stores");
  static_assert(PITCH <= EpiStage<C>::PITCH, "strip too small");
  const uint32_t wbase = lds_strip + (lane % MI) * PITCH + (lane / MI) * (QD::N * sizeof(raw));
  if (gm0 >= m) return;
  const int rows_left = m - gm0 < C::WTM ? (int)(m - gm0) : C::WTM;
  // A bias per row of C (conv2d's 1x1 layers): a lane's row in every row-block is lane % MI.
  constexpr bool WITH_BIAS = BIAS && std::is_same<acc_s, float>::value && !GLU;
  float bias_rows[WITH_BIAS ? C::TM : 1] = {};
  if constexpr (WITH_BIAS) {
    if (bias) bias_of_rows<C::TM, MI>(bias, bias_dtype, (int)gm0, rows_left, lane, bias_rows);
  }
  // this lane's places: row of the row-block, columns of the chunk that exist, strip address, address in C
  int l_row[RP::NL], l_cols[RP::NL];
  uint32_t l_lds[RP::NL];
  raw* l_dst[RP::NL];
#pragma unroll
  for (int t = 0; t < RP::NL; ++t) {
    const int q = t * 64 + lane, row = q / CPRW, cc = q % CPRW;
    const int64_t left = ncols - (gc0 + cc * OUTV);
    const bool idle = MI * CPRW % 64 != 0 && row >= MI;
    l_row[t] = row;
    l_cols[t] = idle || left <= 0 ? 0 : left < OUTV ? (int)left : OUTV;
    l_lds[t] = lds_strip + (idle ? MI - 1 : row) * PITCH + cc * 16;
    l_dst[t] = (raw*)cbase + (gm0 + row) * scm + (gc0 + cc * OUTV) * scn;
  }
  auto put = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int g = 0; g < NGRP; ++g) {
        acc_s v[4] = {acc[i][j][4 * g + 0], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        if constexpr (WITH_BIAS) {                      // added to the finished fp32 sum before the one rounding
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += bias_rows[i];
        }
        // (typed vector store: __builtin_bit_cast on an ext-vector element reads element 0)
        *TNX_LDS(typename QD::vec, wbase + (j * MI + g * 8) * (QD::N * sizeof(raw) / 4)) = QD::run(v[0], v[1], v[2], v[3], epi);
      }
  };
  put(0);
#pragma unroll
  for (int i = 0; i < C::TM; ++i) {
    if (i * MI >= rows_left) break;                     // row-blocks past the last row hold nothing
    // UNR passes from `it0` on: strip reads together, then one store after the other
    auto passes = [&](int it0, auto last) __attribute__((always_inline)) {
      i32x4 v[RP::UNR];
#pragma unroll
      for (int u = 0; u < RP::UNR; ++u)
        v[u] = *TNX_LDS(i32x4, l_lds[RP::EVEN ? 0 : it0 + u] + (RP::EVEN ? (it0 + u) * RP::RSTEP : 0) * PITCH);
      if constexpr (decltype(last)::value)
        if (i + 1 < C::TM) put(i + 1 < C::TM ? i + 1 : i);
#pragma unroll
      for (int u = 0; u < RP::UNR; ++u) {
        const int t = RP::EVEN ? 0 : it0 + u, step = RP::EVEN ? (it0 + u) * RP::RSTEP : 0;
        if (l_row[t] >= rows_left - (i * MI + step) || l_cols[t] == 0) continue;
        raw* dst = l_dst[t] + (int64_t)(i * MI + step) * scm;
        if (vec_ok && l_cols[t] == OUTV) {
          store16_stream_loose(dst, v[u]);              // rows of C need not be 16-byte aligned
        } else {
          raw out[OUTV];
          __builtin_memcpy(out, &v[u], 16);
#pragma unroll 1
          for (int x = 0; x < l_cols[t]; ++x) dst[x * scn] = out[x];
        }
      }
    };
    if constexpr (RP::ITERS == RP::UNR) {
      passes(0, BoolTag<true>{});
    } else if constexpr (RP::EVEN) {
#pragma unroll 1
      for (int it0 = 0; it0 < RP::ITERS; it0 += RP::UNR) passes(it0, BoolTag<false>{});
      if (i + 1 < C::TM) put(i + 1 < C::TM ? i + 1 : i);
    } else {
#pragma unroll
      for (int it0 = 0; it0 < RP::ITERS; it0 += RP::UNR) passes(it0, BoolTag<false>{});
      if (i + 1 < C::TM) put(i + 1 < C::TM ? i + 1 : i);
    }
  }
}

// Epilogue of the persistent kernel.  The ring is already being refilled with the next tile's
// first slabs while this runs, so the accumulators pass through a small strip of their own: per wave
// MI rows x 64 accumulator columns (64 / MI MFMA tiles side by side), rows 256 bytes apart with the
// 16-byte chunk index XOR-ed with the row, so neither the column-wise writes nor
// the row-wise read-back collide on banks.  FULL: the tile lies inside C and C takes 16-byte
// stores, so the number of store instructions per wave is the compile-time STORES (the caller's
// vmcnt arithmetic relies on it).
template <class C> struct PairStrip {
  static constexpr int WAVE_BYTES = C::MI * 256;              // MI rows of 64 accumulator columns
  static constexpr int BYTES = C::NW * WAVE_BYTES;
  static constexpr int TPP = 64 / C::MI;                      // MFMA tiles side by side in one pass
};
template <class T, class C, class O, bool GLU> struct PairEpilogue {
  typedef typename T::acc_s acc_s;
  typedef Pack16<O, acc_s, GLU> PK;
  static constexpr int OCOLS = GLU ? 32 : 64;                 // output columns per pass
  static constexpr int CPRW = OCOLS / PK::OUTV;               // lanes per output row
  static constexpr int ITERS = C::MI * CPRW / 64;
  static constexpr int CH = PK::NF / 4;                       // 16-byte chunks one lane reads back
  static constexpr int STORES = C::TM * (C::TN / PairStrip<C>::TPP) * ITERS;  // store instructions per wave on a FULL tile
};
template <class T, class C, class O, bool GLU, bool FULL, class ACC>
__device__ __forceinline__ void epilogue_store_pairs(ACC (&acc)[C::TM][C::TN], uint8_t* cbase, uint32_t strip, int lane,
                                                     int64_t gm0, int64_t gc0, int64_t m, int64_t ncols, int64_t scm,
                                                     int64_t scn, bool vec_ok, int epi) {
  constexpr int MI = C::MI, TPP = PairStrip<C>::TPP, NGRP = C::ACC_N / 4;
  static_assert(C::TN % TPP == 0 && MI * PairEpilogue<T, C, O, GLU>::CPRW >= 64, "a pass is 64 accumulator columns wide");
  typedef PairEpilogue<T, C, O, GLU> E;
  typedef typename E::acc_s acc_s;
  typedef typename E::PK PK;
  typedef typename PK::raw raw;
  typedef acc_s acc4 __attribute__((ext_vector_type(4)));
  raw* cp = (raw*)cbase;
  const int wrow = lane % MI, wk = lane / MI;
  const uint32_t wbase = strip + wrow * 256;
#pragma unroll
  for (int i = 0; i < C::TM; ++i) {
    if (!FULL && gm0 + i * MI >= m) break;
#pragma unroll
    for (int jp = 0; jp < C::TN / TPP; ++jp) {
#pragma unroll
      for (int jj = 0; jj < TPP; ++jj)
#pragma unroll
        for (int g = 0; g < NGRP; ++g) {
          // chunk of four columns inside the 64-column pass: tile jj, then the lane's column group
          const int c = jj * (MI / 4) + g * (64 / MI) + wk;
          *TNX_LDS(acc4, wbase + ((c ^ (wrow & 15)) << 4)) =
              acc4{acc[i][TPP * jp + jj][4 * g + 0], acc[i][TPP * jp + jj][4 * g + 1], acc[i][TPP * jp + jj][4 * g + 2],
                   acc[i][TPP * jp + jj][4 * g + 3]};
        }
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the strip is private to the wave
      acc_s f[E::ITERS][PK::NF];
#pragma unroll
      for (int it = 0; it < E::ITERS; ++it) {
        const int q = it * 64 + lane;
        const int row = q / E::CPRW, cc = q % E::CPRW;
#pragma unroll
        for (int x = 0; x < E::CH; ++x) {
          const i32x4 v = *TNX_LDS(i32x4, strip + row * 256 + (((cc * E::CH + x) ^ (row & 15)) << 4));
          __builtin_memcpy(&f[it][4 * x], &v, 16);
        }
      }
#pragma unroll
      for (int it = 0; it < E::ITERS; ++it) {
        const int q = it * 64 + lane;
        const int row = q / E::CPRW, cc = q % E::CPRW;
        const int64_t gm = gm0 + i * MI + row;
        const int64_t gc = gc0 + jp * E::OCOLS + cc * PK::OUTV;
        raw out[PK::OUTV];
        PK::run(f[it], epi, out);
        raw* dst = cp + gm * scm + gc * scn;
        if (FULL) {
          i32x4 v;
          __builtin_memcpy(&v, out, 16);
          store16_stream(dst, v);
        } else if (gm < m) {
          if (vec_ok && gc + PK::OUTV <= ncols) {
            i32x4 v;
            __builtin_memcpy(&v, out, 16);
            store16_stream(dst, v);
          } else {
#pragma unroll 1
            for (int x = 0; x < PK::OUTV; ++x)
              if (gc + x < ncols) dst[x * scn] = out[x];
          }
        }
      }
      __builtin_amdgcn_s_waitcnt(0xC07F);  // the next pass overwrites the strip
    }
  }
}

// The first WS_COUNTER_BYTES of the split-K workspace hold one arrival counter per cut tile.
// They must be zero when a launch starts; every launch leaves them zero.
constexpr int WS_COUNTER_BYTES = 65536;
constexpr int WS_MAX_TILES = WS_COUNTER_BYTES / 4;

// One K slice of a cut tile leaves the workgroup: every wave writes its accumulators to its
// part of the slice with device-scope (sc1) stores, one lane bumps the tile's arrival counter,
// and the function returns true in the workgroup that arrived last.  That workgroup then reads
// all slices back with device-scope loads and runs the ordinary epilogue on their sum.
// Whole-L2 write-backs and invalidates (what a device-scope fence costs on a part with eight
// L2s) are avoided on purpose: they cost more than the GEMM.
// FLAG_APART: the flag's LDS word is not part of the epilogue strips that are written next.
template <class T, class C, bool FLAG_APART, class ACC>
__device__ __forceinline__ bool splitk_arrive(ACC (&acc)[C::TM][C::TN], uint8_t* wave_slice, int lane, int64_t gm0, int64_t m,
                                              int* counter, int* flag, int nslices, bool atomic) {
  typedef typename T::acc_s acc_s;
  typedef acc_s acc4 __attribute__((ext_vector_type(4)));
  constexpr int NGRP = C::ACC_N / 4;
  constexpr int NQ = C::TN * NGRP;                      // 16-byte groups per lane and row-block
  const __amdgpu_buffer_rsrc_t win = agent_window(wave_slice);
#pragma unroll
  for (int i = 0; i < C::TM; ++i) {
    if (gm0 + i * C::MI >= m) break;
    if (gm0 + i * C::MI + lane % C::MI >= m) continue;   // a lane is one row: rows past the problem are not stored
    if (atomic) {
      // every slice adds into the same copy (wave_slice is slice 0 for all of them); same element order as a stored slice
      acc_s* dst = (acc_s*)(wave_slice + (int64_t)i * NQ * 1024 + lane * 16);
#pragma unroll
      for (int j = 0; j < C::TN; ++j)
#pragma unroll
        for (int g = 0; g < NGRP; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            __hip_atomic_fetch_add(dst + (j * NGRP + g) * 256 + e, acc[i][j][4 * g + e], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    } else {
#pragma unroll
      for (int j = 0; j < C::TN; ++j)
#pragma unroll
        for (int g = 0; g < NGRP; ++g) {
          const acc4 v = {acc[i][j][4 * g + 0], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
          i32x4 w;
          __builtin_memcpy(&w, &v, 16);
          store16_agent(win, (uint32_t)lane * 16u + (uint32_t)(i * NQ + j * NGRP + g) * 1024u, w);
        }
    }
  }
  // device-scope stores: once they are acknowledged they are visible to every XCD, so the
  // arrival count may follow
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int prev = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the last arrival re-arms the counter for the next launch
    if (prev == nslices - 1) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = prev;
  }
  __syncthreads();
  const bool last = *flag == nslices - 1;
  if constexpr (!FLAG_APART) __syncthreads();
  return last;
}

// 16 bytes from an address that is only 2-byte aligned
struct __attribute__((packed, aligned(2))) Loose16 {
  i32x4 v;
};


// Epilogue of the CONV kernels: rows are output channels, columns are pixels of the padded pixel index space.  Same
// pass through the wave's LDS strip as epilogue_store; a chunk is 8 pixels of one output row, so it is one
// run of the NCHW output (cut at w_out: the pixels past it exist only in the index space).  Bias is added in fp32; it is
// fetched up front (a load per row-block in the middle of the loop put a memory round trip on each of up to eight), and
// a chunk's place in the output is worked out once per lane.
template <class T, class C, class O, class ACC>
__device__ __forceinline__ void epilogue_store_conv(ACC (&acc)[C::TM][C::TN], uint8_t* ybase, uint32_t lds_strip, int lane,
                                                    int gm0, int gn0, const ConvGeom& g) {
  typedef Quad<O, float, false> QD;
  typedef typename O::raw raw;                          // 16-bit outputs, or binary32 (the fp32 sums + bias as they are)
  constexpr int MI = C::MI;
  constexpr int NGRP = C::ACC_N / 4;
  constexpr int PITCH = C::WTN * sizeof(raw) + 16;
  constexpr int CPRW = C::WTN / 8;                       // a lane handles 8 pixels: one 16-byte chunk of the im2col slab
  typedef RowPasses<MI, CPRW> RP;
  static_assert(PITCH <= EpiStage<C>::PITCH && C::WTN % 8 == 0 && RP::ITERS == RP::UNR, "one row-block per pass, 8 outputs per chunk");
  const uint32_t wbase = lds_strip + (lane % MI) * PITCH + (lane / MI) * (4 * sizeof(raw));
  if (gm0 >= g.c_out) return;
  const int rows_left = g.c_out - gm0 < C::WTM ? g.c_out - gm0 : C::WTM;
  float bias_rows[C::TM] = {};
  if (g.bias) bias_of_rows<C::TM, MI>(g.bias, g.bias_dtype, gm0, rows_left, lane, bias_rows);
  const int64_t plane = (int64_t)g.h_out * g.w_out;
  // this lane's places: row of the row-block, pixels of the chunk that exist, strip address, address in the output
  int l_row[RP::NL], l_valid[RP::NL];
  uint32_t l_lds[RP::NL];
  raw* l_dst[RP::NL];
#pragma unroll
  for (int t = 0; t < RP::NL; ++t) {
    const int q = t * 64 + lane, row = q / CPRW, cc = q % CPRW;
    const bool idle = MI * CPRW % 64 != 0 && row >= MI;
    const int gc = gn0 + cc * 8;
    const int img = (int)fd_div((uint32_t)gc, g.div_hwp);
    const int r = gc - img * (g.h_out * g.wp);
    const int ho = (int)fd_div((uint32_t)r, g.div_wp);
    const int wq = r - ho * g.wp;
    const int valid = g.w_out - wq;                     // pixels of this chunk that exist
    l_row[t] = row;
    l_valid[t] = idle || gc >= g.n_total || valid <= 0 ? 0 : valid < 8 ? valid : 8;
    l_lds[t] = lds_strip + (idle ? MI - 1 : row) * PITCH + cc * (8 * sizeof(raw));
    l_dst[t] = (raw*)ybase + ((int64_t)img * g.c_out + gm0 + row) * plane + (int64_t)ho * g.w_out + wq;
  }
  auto put = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < C::TN; ++j)
#pragma unroll
      for (int q = 0; q < NGRP; ++q)
        *TNX_LDS(typename QD::vec, wbase + (j * MI + q * 8) * sizeof(raw)) =
            QD::run(acc[i][j][4 * q + 0] + bias_rows[i], acc[i][j][4 * q + 1] + bias_rows[i], acc[i][j][4 * q + 2] + bias_rows[i],
                    acc[i][j][4 * q + 3] + bias_rows[i], 0);
  };
  put(0);
#pragma unroll
  for (int i = 0; i < C::TM; ++i) {
    if (i * MI >= rows_left) break;
    constexpr int H = sizeof(raw) / 2;                  // 16-byte halves of a chunk
    i32x4 v[RP::UNR][H];
#pragma unroll
    for (int u = 0; u < RP::UNR; ++u)
#pragma unroll
      for (int h = 0; h < H; ++h) v[u][h] = *TNX_LDS(i32x4, l_lds[RP::EVEN ? 0 : u] + (RP::EVEN ? u * RP::RSTEP : 0) * PITCH + 16 * h);
    if (i + 1 < C::TM) put(i + 1 < C::TM ? i + 1 : i);
#pragma unroll
    for (int u = 0; u < RP::UNR; ++u) {
      const int t = RP::EVEN ? 0 : u, step = RP::EVEN ? u * RP::RSTEP : 0;
      if (l_row[t] >= rows_left - (i * MI + step) || l_valid[t] == 0) continue;
      raw* dst = l_dst[t] + (int64_t)(i * MI + step) * plane;
      if (l_valid[t] == 8) {
#pragma unroll
        for (int h = 0; h < H; ++h) {                   // element-aligned: w_out need not be a multiple of 8
          // binary32: the two stores of a lane interleave with its neighbours', so each fills half of every cache line;
          // kept in the L2 the halves meet there, hinted they go out one by one (1984 channels of 17x17, batch 64:
          // 116 -> 64 us)
          if constexpr (H == 2) *(i32x4_loose*)((uint8_t*)dst + 16 * h) = v[u][h];
          else store16_stream_loose(dst, v[u][h]);
        }
      } else {
        raw out[8];
        __builtin_memcpy(out, v[u], 8 * sizeof(raw));
#pragma unroll 1
        for (int x = 0; x < l_valid[t]; ++x) dst[x] = out[x];
      }
    }
  }
}

// GATHER: the table of k-chunk offsets behind the ring
constexpr int GATHER_TABLE_BYTES = 8192;

// ---------------------------------------------------------------------------
// the kernel
// ---------------------------------------------------------------------------
// BT: B is k-contiguous (element (k, n) at b + n * stride_bn + k, the layout of `x @ w.t()` with a
// row-major weight): its slab sits in LDS as BN rows of BK elements exactly like the A slab, and its
// fragments are read with plain ds_read_b128 -- no transposing read is needed.
// CONV: conv2d forward (ConvGeom): A is the weight, the B slab is gathered from the NCHW input by the DMA loader --
// one 16-byte raw-buffer load per chunk of 8 pixels from an address that is only 2-byte aligned, with an
// out-of-range offset (the buffer bound answers zero) for chunks whose input row lies in the padding.  The elements
// of a chunk that fall into the left / right padding have to be zeroed in LDS afterwards, by the wave that loaded
// them.  Done between the wait for the loads and the barrier that publishes the slab, that fix-up sits on the
// critical path of every K slab (measured: 340 instead of 630 TFLOP/s on a 3x3 layer), so the ring has three slots
// and a slab is fixed well before it is read: slab t+3 is issued during the first half of period t, waited for in
// the middle of period t+1 (by then only that period's own loads may still be outstanding), fixed in the second
// half of period t+1 -- one read-modify-write of the chunk per op, slotted behind MFMAs -- and published by barrier
// t+2, before whose period nothing reads it.  16-bit types, stride_w == 1, k % BK == 0.
// AT: A is m-contiguous (element (m, k) at a + k * stride_ak + m, the layout of `x.t() @ dy`): its slab sits in LDS as
// BK rows of BM elements exactly like a row-major B slab, and its fragments are read with the transposing reads.
// PAIR: a float32 product.  A K slab of 64 holds the bf16 heads of 32 k (k step 0) and their tails (k step 1), and each
// slab takes three MFMA steps from these two fragment sets -- head head, tail head, head tail -- where three copies laid
// along k would read six; the result is binary32.  (Kernels of their own: a second epilogue and loop in one kernel cost
// the 192- and 256-wide tiles hundreds of spilled registers.)
// GATHER (with BT): conv2d forward over a packed input (PackGeom): the rows of the k-contiguous B slab are the windows of
// BN output pixels.  A lane's DMA ops fetch the same 16-byte k chunk of different pixels, so an op's offset is the
// pixel's, kept in a register, plus the chunk's (filter tap, channels), read once per slab from a table in LDS.  Chunks
// past the end of k get an offset outside the buffer and arrive as zeros.
template <class T, class C, bool FAST, bool PERSIST = false, bool BT = false, bool CONV = false, bool GATHER = false, bool AT = false, bool PAIR = false>
__global__ __launch_bounds__(C::THREADS, PERSIST ? 1 : Residency<C>::WAVES) void gemm_tile_kernel(typename KernelParams<FAST && !CONV && !GATHER>::type in) {
  GemmParams p;
  if constexpr (FAST && !CONV && !GATHER) p = expand_params<C, BT, AT>(in);
  else p = in;
  constexpr int ES = C::ES, BM = C::BM, BN = C::BN, BK = C::BK, NW = C::NW, STAGES = C::STAGES;
  constexpr int MI = C::MI, TM = C::TM, TN = C::TN;
  static_assert(GATHER ? C::VALID_GATHER : C::VALID, "tile configuration not supported by this kernel");
  static_assert(!GATHER || (FAST && BT && !PERSIST && !CONV), "the packed conv2d variant is a k-contiguous-B kernel");
  static_assert(!AT || (FAST && !PERSIST && !BT && !CONV && C::VALID_AT), "the m-contiguous A variant is built with the DMA loader, row-major B");
  static_assert(!PERSIST || FAST, "the persistent kernel is built with the DMA loader only");
  static_assert(!BT || (FAST && (GATHER || C::B_LOADS % NW == 0)), "the k-contiguous B variant is built with the DMA loader only");
  static_assert(!CONV || (FAST && !PERSIST && !BT && ES == 2 && STAGES == 3 && MI == 16 && (NW * 64) % C::CPR_B == 0),
                "the conv2d variant: DMA loader, 16-bit types, three ring slots");
  static_assert(!PAIR || (FAST && !PERSIST && !CONV && C::KSTEPS == 2 && C::MMA_K == 32), "the float32 variant: DMA loader, slabs of 32 heads and 32 tails");
  typedef Mma<T, MI> MMA;
  typedef typename MMA::acc_t acc_t;
  typedef typename T::acc_s acc_s;
  // Several problems in one grid and a bias per row (GemmParams::batch, cv.bias) exist in the tiles up to 128x128:
  // the 256-wide tiles have no register to spare for the extra state (measured: 20 more spilled registers, -0.4 %).
  constexpr bool MULTI = !PERSIST && !CONV && !GATHER && !PAIR && multi_problem_tile<C>();

  constexpr int AT_CPR = BM * ES / 16, AT_ROWB = BM * ES;    // AT: chunks and bytes of an A slab row

  // one workgroup per tile: the epilogue strips are laid over the ring once the K loop is done.
  // persistent: the ring is refilled for the next tile during the epilogue, so the strips follow it.
  constexpr int RING_OR_STRIPS = C::LDS_BYTES > EpiStage<C>::BYTES ? C::LDS_BYTES : EpiStage<C>::BYTES;
  // CONV: behind the ring, a table of the 81 16-byte masks that keep elements [lo, hi) of a chunk (0 <= lo, hi <= 8),
  // and two tables of the filter taps of one K slab (BK entries of 8 bytes: element offset, dh | dw << 16)
  constexpr int CV_TABLE_BYTES = CONV ? 81 * 16 + 2 * BK * 8 : 0;
  constexpr int SMEM_BYTES = (PERSIST ? C::LDS_BYTES + PairStrip<C>::BYTES : RING_OR_STRIPS) + CV_TABLE_BYTES +
                             (GATHER ? GATHER_TABLE_BYTES : 0);
  static_assert(SMEM_BYTES <= 163840, "LDS budget of one CU exceeded");
  __shared__ __attribute__((aligned(1024))) uint8_t smem[SMEM_BYTES];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(uint8_t __attribute__((address_space(3)))*)smem;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- which tile / split ------------------------------------------------
  // Tiles [0, split_tile0) in launch order are computed whole by one workgroup each; the
  // tiles after them are cut split_k ways along K (all tiles when split_tile0 == 0: plain
  // split-K; only the last partial wave of tiles when the tile count does not fill the CUs).
  // The persistent kernel never cuts: workgroup b computes tiles b, b + gridDim.x, ... whole.
  const int ntiles = p.tiles_m * p.tiles_n;
  int split = 0, logical = 0;
  bool cut = false;
  // launch-order id -> tile coordinates
  auto locate = [&](int id, int* pid_m, int* pid_n) __attribute__((always_inline)) {
    if (p.tile_order == 1) {
      superblock_order(id, p.tiles_m, p.tiles_n, pid_m, pid_n);
    } else {
      const int lg = xcd_remap(id, ntiles, 8);
      swizzle2d(lg, p, pid_m, pid_n);
    }
  };
  int pid_m, pid_n;
  if (PERSIST || p.split_k <= 1) {
    int bid = blockIdx.x;
    if constexpr (MULTI) {
      // several problems with one A in one grid (conv2d's 1x1 layers: one per image): problem after problem
      if (p.batch > 1) {
        const int img = (int)fd_div((uint32_t)bid, p.div_tiles);
        bid -= img * ntiles;
        p.b += (int64_t)img * p.b_batch_bytes;
        p.c += (int64_t)img * p.c_batch_bytes;
      }
    }
    locate(bid, &pid_m, &pid_n);
  } else {
    if ((int)blockIdx.x < p.split_tile0) {
      logical = xcd_remap(blockIdx.x, p.split_tile0, 8);
    } else {
      const int ncut = ntiles - p.split_tile0;
      int t = blockIdx.x - p.split_tile0;
      split = (int)fd_div((uint32_t)t, p.div_cut);
      t -= split * ncut;
      logical = p.split_tile0 + xcd_remap(t, ncut, 8);
      cut = true;
    }
    swizzle2d(logical, p, &pid_m, &pid_n);
  }

  const int kt_total = (int)((p.k + BK - 1) / BK);
  const int kt0 = cut ? split * p.ktiles_per_split : 0;
  int kt1 = cut ? kt0 + p.ktiles_per_split : kt_total;
  if (kt1 > kt_total) kt1 = kt_total;
  // FAST kernels move their slabs with the DMA loader.  It wants chunks that lie inside their row: with a K that is
  // no multiple of BK, rows that are not 16-byte aligned or an N that ends inside a chunk, the host sets tail_slab
  // and the last slab of the K range (the only one whose chunks can cross the end of a row of A, or the end of the
  // last row of B) is left out of the ring and fetched after the K loop (load_tail).  Past k it then holds zeros; columns past n, or
  // rows past m of an m-contiguous A, hold whatever follows them and must never be stored.
  const bool tail_here = FAST && !PERSIST && !CONV && !GATHER && !PAIR && p.tail_slab != 0 && kt1 == kt_total && kt1 > kt0;
  const int KT = kt1 > kt0 ? kt1 - kt0 - (tail_here ? 1 : 0) : 0;          // slabs of this workgroup in the ring (per tile)

  // ---- the tile the loader works on: origin, DMA bases and per-lane byte offsets.
  // (In the persistent kernel the loader moves on to the next tile before the epilogue of the
  // current one has run, so the epilogue keeps its own copy of the origin.)
  int64_t m0 = 0, n0 = 0;
  uint32_t a_voff[C::A_LPW], b_voff[C::B_LPW];
  constexpr bool PINGPONG_TILE = TNX_PINGPONG && FAST && !PERSIST && !BT && !CONV && NW == 8 && STAGES == 2 && C::KSTEPS == 2;
  // CONV: a lane's B ops all fetch the same 16-byte LDS column slot; the pixel chunk that lands there is one of
  // two (the LDS swizzle moves it by two chunks depending on the k row): element offset of (image, channel 0,
  // h0, w0) and the packed (h0, w0) for both, (h0, w0) being the input position of filter tap (0, 0).  Pixels past
  // the end get h0 = -32768, which no tap brings back into the image.  The filter taps (dh, dw, element offset) of
  // the k rows of a slab come from a 64-entry table in LDS that the first 64 threads write one period ahead, each
  // keeping the running tap of one k row and moving it one slab on per period (additions and wrap-arounds only):
  // per op a lane reads one entry instead of doing that arithmetic itself.
  constexpr int CONV_STEP = (NW * 64) / C::CPR_B;          // k rows covered by one B op of the workgroup
  const int cv_r0 = tid / C::CPR_B;                          // k row of this lane in the first op of a slab
  int pix_off0 = 0, pix_off1 = 0, pix_hw0 = 0, pix_hw1 = 0;   // (scalars, not arrays: an array indexed by a run-time bit is moved to LDS by the compiler)
  int tap_dh = 0, tap_dw = 0;                                // (wave 0 only) tap of k row `tid` of the next slab to tabulate
  uint32_t tap_off = 0;
  int cv_wr = 0, cv_rd = 0;                                  // next slab to tabulate / to issue (their parities pick the table)
  i32x2 cv_ent[CONV ? C::B_LPW : 1];                         // the table entries of this lane's ops of the slab being issued
  uint32_t cv_fix[CONV ? C::B_LPW : 1];                      // per op of the slab in flight: what its fix-up has to do
  int cv_o[CONV ? C::B_LPW : 1];                             // ... and the element offset its chunk starts at
  bool cv_pending = false;
  uint32_t cv_dst = 0;
  constexpr uint32_t CV_OUTSIDE = 0xffffffffu, CV_NOFIX = 8u * 16u;   // a note is the byte offset of mask (lo, hi) in the table: (lo * 9 + hi) * 16
  const uint32_t cv_table = lds0 + RING_OR_STRIPS;
  const uint32_t cv_ktab = cv_table + 81 * 16;
  i32x4 cv_rsrc = {0, 0, 0, 0};
  if constexpr (CONV) {
    if (tid < 81) {
      const int lo = tid / 9, hi = tid % 9;
      i32x4 m;
#pragma unroll
      for (int d = 0; d < 4; ++d)
        m[d] = (int)((2 * d >= lo && 2 * d < hi ? 0xffffu : 0u) | (2 * d + 1 >= lo && 2 * d + 1 < hi ? 0xffff0000u : 0u));
      *TNX_LDS(i32x4, cv_table + tid * 16) = m;
    }
    __syncthreads();
    const uint64_t xa = (uint64_t)(uintptr_t)p.b;
    cv_rsrc = i32x4{(int)__builtin_amdgcn_readfirstlane((uint32_t)xa), (int)(__builtin_amdgcn_readfirstlane((uint32_t)(xa >> 32)) & 0xffff),
                    (int)__builtin_amdgcn_readfirstlane(p.cv.x_bytes), 0x00020000};
  }
  // GATHER: chunk offsets of this workgroup's K range: one entry per chunk, or per slab when a filter tap's channels are
  // whole slabs (the chunk's place in the slab is then part of the pixel offset).  All chunks a lane fetches have the
  // same place in their slab: the swizzle of a row depends on the row modulo 8, which is lane / 8.
  const uint32_t g_table = lds0 + RING_OR_STRIPS;
  const int g_chunk = (lane & 7) ^ C::swzA(lane >> 3);
  const bool g_whole = GATHER && p.pk.cpt % 8 == 0;
  uint32_t g_at = g_table + (g_whole ? 0 : g_chunk * 4);     // entry of the next slab to issue
  uint32_t g_tap = 0;                                        // offset of the slab being issued
  i32x4 g_rsrc = {0, 0, 0, 0};
  if constexpr (GATHER) {
    const PackGeom& g = p.pk;
    const int ents = g_whole ? kt1 - kt0 : (kt1 - kt0) * 8;
    for (int e = tid; e < ents; e += C::THREADS) {
      const int k8 = kt0 * 8 + (g_whole ? e * 8 : e);
      int tap, c8;
      if (g_whole) {        // slabs of 64 channels, the filter taps of one slab after another
        const int cs = (int)fd_div((uint32_t)(kt0 + e), g.div_taps);
        tap = kt0 + e - cs * g.taps;
        c8 = cs * 8;
      } else {
        tap = (int)fd_div((uint32_t)k8, g.div_cpt);
        c8 = k8 - tap * g.cpt;
      }
      const int r = (int)fd_div((uint32_t)tap, g.div_fw), s = tap - r * g.fw;
      const uint32_t off = (uint32_t)r * g.tap_row_bytes + (uint32_t)s * g.tap_col_bytes + (uint32_t)c8 * 16u;
      *TNX_LDS(uint32_t, g_table + e * 4) = k8 < g.chunks ? off : 0x80000000u;
    }
    const uint64_t xa = (uint64_t)(uintptr_t)p.b;
    g_rsrc = i32x4{(int)__builtin_amdgcn_readfirstlane((uint32_t)xa), (int)(__builtin_amdgcn_readfirstlane((uint32_t)(xa >> 32)) & 0xffff),
                   (int)__builtin_amdgcn_readfirstlane(g.x_bytes), 0x00020000};
  }
  const uint8_t* a_sbase = p.a;
  const uint8_t* b_sbase = p.b;
  // DMA op q of this wave moves 1 KiB number b_op(q) of the B slab
  auto b_op = [&](int q) __attribute__((always_inline)) {
    const int op = q * NW + wave;
    return C::B_LOADS % NW != 0 && op >= C::B_LOADS ? C::B_LOADS - 1 : op;
  };
  auto place_tile = [&](int tile_m, int tile_n) __attribute__((always_inline)) {
    m0 = (int64_t)tile_m * BM;
    n0 = (int64_t)tile_n * BN;
    if (FAST) {
      const int64_t lda = p.sam, ldb = BT ? p.sbn : p.sbk;
      // wave-uniform by construction; say so, so both stay in SGPRs for the DMA's scalar base operand
      a_sbase = uniform_ptr(AT ? p.a + ((int64_t)kt0 * BK * p.sak + m0) * ES : p.a + (m0 * lda + (int64_t)kt0 * BK) * ES);
      b_sbase = uniform_ptr(BT ? p.b + (n0 * ldb + (int64_t)kt0 * BK) * ES : p.b + ((int64_t)kt0 * BK * ldb + n0) * ES);
      const int64_t mrem = p.m - 1 - m0;  // last valid row inside this tile
#pragma unroll
      for (int q = 0; q < C::A_LPW; ++q) {
        int P = (q * NW + wave) * 64 + lane;
        if constexpr (AT) {
          // rows of the slab are k, as in a row-major B slab: chunks past M as chunks past N there
          int row = P / AT_CPR, cs = P % AT_CPR;
          int c = cs ^ C::template swzT<AT_CPR>(row);
          if (m0 + (int64_t)c * (16 / ES) >= p.m_load || (!p.tail_slab && m0 + (int64_t)(c + 1) * (16 / ES) > p.m_load)) c = 0;
          a_voff[q] = (uint32_t)((int64_t)row * p.sak * ES + c * 16);
          continue;
        }
        int row = P / C::CPR_A, cs = P % C::CPR_A;
        int c = cs ^ C::swzA(row);
        int64_t r = row < mrem ? row : mrem;
        a_voff[q] = (uint32_t)(r * lda * ES + c * 16);
      }
      if constexpr (CONV) {
        const ConvGeom& g = p.cv;
        const int cs = tid % C::CPR_B;
        const int c0 = cs ^ C::swzB(cv_r0 & 7);              // rows 0-7: the swizzle without its pass term
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const int n = (int)n0 + ((c0 ^ (v << 1)) << 3);
          int off = 0, h0 = -32768, w0 = 0;
          if (n < g.n_total) {
            const int img = (int)fd_div((uint32_t)n, g.div_hwp);
            const int r = n - img * (g.h_out * g.wp);
            const int ho = (int)fd_div((uint32_t)r, g.div_wp);
            h0 = ho * g.stride_h - g.pad_h;
            w0 = (r - ho * g.wp) - g.pad_w;
            off = img * g.chw_in + h0 * g.w_in + w0;
          }
          const int hw = (int)(((uint32_t)h0 << 16) | ((uint32_t)w0 & 0xffffu));
          if (v == 0) { pix_off0 = off; pix_hw0 = hw; } else { pix_off1 = off; pix_hw1 = hw; }
        }
        // the tap of k row tid (< BK) of slab 0 (the K loop starts at k = 0: these kernels are never cut along K)
        const int krow = tid & (BK - 1);
        const int cin = (int)fd_div((uint32_t)krow, g.div_rs);
        const int r = krow - cin * g.rs;
        const int th = (int)fd_div((uint32_t)r, g.div_s);
        tap_dh = th * g.dil_h;
        tap_dw = (r - th * g.fw) * g.dil_w;
        tap_off = (uint32_t)(cin * g.hw_in + tap_dh * g.w_in + tap_dw);
        cv_wr = 0;
        cv_rd = 0;
      }
      const int64_t nrem = p.n - 1 - n0;  // last valid column inside this tile
#pragma unroll
      for (int q = 0; q < (CONV ? 0 : C::B_LPW); ++q) {
        int P = (q * NW + wave) * 64 + lane;
        if constexpr (GATHER) {
          const PackGeom& g = p.pk;
          int n = (int)n0 + b_op(q) * 8 + (lane >> 3);
          n = n < p.cv.n_total ? n : p.cv.n_total - 1;          // pixels past the end are computed and dropped
          const int img = (int)fd_div((uint32_t)n, g.div_hwp);
          int r = n - img * g.hwp;
          r = r < g.hw_out ? r : g.hw_out - 1;
          const int ho = (int)fd_div((uint32_t)r, g.div_w), wo = r - ho * g.w_out;
          b_voff[q] = (uint32_t)img * g.img_bytes + (uint32_t)ho * g.row_bytes + (uint32_t)wo * g.col_bytes +
                      (g_whole ? (uint32_t)g_chunk * 16u : 0u);
        } else if (BT) {
          // rows of the slab are columns of B: same chunk layout and swizzle as the A slab
          int row = P / C::CPR_A, cs = P % C::CPR_A;
          int c = cs ^ C::swzA(row);
          int64_t r = row < nrem ? row : nrem;
          b_voff[q] = (uint32_t)(r * ldb * ES + c * 16);
        } else {
          int row = P / C::CPR_B, cs = P % C::CPR_B;
          int c = cs ^ C::swzB(row);
          // column chunk past N: any valid address.  (A chunk that starts below N and ends above it -- tail_slab
          // launches only -- is loaded as it is: its upper elements come from the k rows after it, which reach that far
          // because the last slab is not loaded here (ring_chunks_inside), and belong to columns that are never stored.)
          if (n0 + (int64_t)c * (16 / ES) >= p.n_load || (!p.tail_slab && n0 + (int64_t)(c + 1) * (16 / ES) > p.n_load)) c = 0;
          b_voff[q] = (uint32_t)((int64_t)row * ldb * ES + c * 16);
        }
      }
    }
  };
  place_tile(pid_m, pid_n);

  // Loader for what the DMA path does not take: any strides, any ragged edge, zero fill.  One 16-byte chunk of the
  // slab per thread and trip: a chunk that lies inside the matrix along a unit-stride dimension is one vector load
  // at the element's own alignment, any other chunk is put together element by element.  Used for every slab of the
  // kernels built without the DMA loader and for the left-out last slabs that load_tail hands on.
  // (t0: the thread's index in the workgroup, handed in so that the DMA kernels need not keep threadIdx.x alive
  // across their K loop for the one call after it)
  // The loader in two halves, so that the kernels built without the DMA loader can fetch slab t + STAGES into
  // registers before the MFMAs of a period and put it into LDS after them (gen_fetch, gen_store).
  constexpr int GEN_B_ROWS = BT ? BN : BK, GEN_B_CPR = BT ? C::CPR_A : C::CPR_B;
  constexpr int GEN_NA = (BM * C::CPR_A + C::THREADS - 1) / C::THREADS;
  constexpr int GEN_NB = (GEN_B_ROWS * GEN_B_CPR + C::THREADS - 1) / C::THREADS;
  typedef std::conditional_t<ES == 4, uint32_t, std::conditional_t<ES == 2, uint16_t, uint8_t>> gen_elem_t;
  typedef std::conditional_t<ES == 4, i32x4_words, std::conditional_t<ES == 2, i32x4_loose, i32x4_bytes>> gen_chunk_t;
  constexpr int EPC = 16 / ES;                           // elements per chunk
  // chunk idx of the A part of slab kt_global: row idx / CPR_A, k chunk idx % CPR_A
  auto gen_fetch_a = [&](int kt_global, int idx) __attribute__((always_inline)) -> i32x4 {
    const gen_elem_t* ap = (const gen_elem_t*)p.a;
    i32x4 v = {0, 0, 0, 0};
    if constexpr (AT) {
      const int64_t gk = (int64_t)kt_global * BK + idx / AT_CPR, gm = m0 + (int64_t)(idx % AT_CPR) * EPC;
      if (idx < BK * AT_CPR && gk < p.k && gm < p.m) {
        if (p.sam == 1 && gm + EPC <= p.m) {
          v = *(const gen_chunk_t*)(ap + gk * p.sak + gm);
        } else {
          gen_elem_t e[EPC];
#pragma unroll
          for (int x = 0; x < EPC; ++x) e[x] = gm + x < p.m ? ap[gk * p.sak + (gm + x) * p.sam] : (gen_elem_t)0;
          __builtin_memcpy(&v, e, 16);
        }
      }
      return v;
    }
    const int row = idx / C::CPR_A, cs = idx % C::CPR_A;
    const int64_t gm = m0 + row, gk = (int64_t)kt_global * BK + cs * EPC;
    if (idx < BM * C::CPR_A && gm < p.m && gk < p.k) {
      if (p.sak == 1 && gk + EPC <= p.k) {
        v = *(const gen_chunk_t*)(ap + gm * p.sam + gk);
      } else {
        gen_elem_t e[EPC];
#pragma unroll
        for (int x = 0; x < EPC; ++x) e[x] = gk + x < p.k ? ap[gm * p.sam + (gk + x) * p.sak] : (gen_elem_t)0;
        __builtin_memcpy(&v, e, 16);
      }
    }
    return v;
  };
  // chunk idx of the B part: k row idx / CPR_B, column chunk idx % CPR_B -- or, for the k-contiguous-B kernels, whose
  // slab holds BN rows of B^T chunked and swizzled like the A slab, column idx / CPR_A, k chunk idx % CPR_A
  auto gen_fetch_b = [&](int kt_global, int idx) __attribute__((always_inline)) -> i32x4 {
    const gen_elem_t* bp = (const gen_elem_t*)p.b;
    const int row = idx / GEN_B_CPR, cs = idx % GEN_B_CPR;
    const int64_t k0 = (int64_t)kt_global * BK;
    i32x4 v = {0, 0, 0, 0};
    if constexpr (BT) {
      const int64_t gn = n0 + row, gk = k0 + cs * EPC;
      if (idx < GEN_B_ROWS * GEN_B_CPR && gn < p.n && gk < p.k) {
        if (p.sbk == 1 && gk + EPC <= p.k) {
          v = *(const gen_chunk_t*)(bp + gn * p.sbn + gk);
        } else {
          gen_elem_t e[EPC];
#pragma unroll
          for (int x = 0; x < EPC; ++x) e[x] = gk + x < p.k ? bp[gn * p.sbn + (gk + x) * p.sbk] : (gen_elem_t)0;
          __builtin_memcpy(&v, e, 16);
        }
      }
    } else {
      const int64_t gk = k0 + row, gn = n0 + cs * EPC;
      if (idx < GEN_B_ROWS * GEN_B_CPR && gk < p.k && gn < p.n) {
        if (p.sbn == 1 && gn + EPC <= p.n) {
          v = *(const gen_chunk_t*)(bp + gk * p.sbk + gn);
        } else {
          gen_elem_t e[EPC];
#pragma unroll
          for (int x = 0; x < EPC; ++x) e[x] = gn + x < p.n ? bp[gk * p.sbk + (gn + x) * p.sbn] : (gen_elem_t)0;
          __builtin_memcpy(&v, e, 16);
        }
      }
    }
    return v;
  };
  auto gen_store_a = [&](uint32_t stage_base, int idx, i32x4 v) __attribute__((always_inline)) {
    if constexpr (AT) {
      const int row = idx / AT_CPR, cs = idx % AT_CPR;
      if (idx < BK * AT_CPR) *TNX_LDS(i32x4, stage_base + row * AT_ROWB + ((cs ^ C::template swzT<AT_CPR>(row)) << 4)) = v;
      return;
    }
    const int row = idx / C::CPR_A, cs = idx % C::CPR_A;
    if (idx < BM * C::CPR_A) *TNX_LDS(i32x4, stage_base + row * C::ROWB_A + ((cs ^ C::swzA(row)) << 4)) = v;
  };
  auto gen_store_b = [&](uint32_t stage_base, int idx, i32x4 v) __attribute__((always_inline)) {
    const int row = idx / GEN_B_CPR, cs = idx % GEN_B_CPR;
    if (idx < GEN_B_ROWS * GEN_B_CPR) {
      if constexpr (BT) *TNX_LDS(i32x4, stage_base + C::A_BYTES + row * C::ROWB_A + ((cs ^ C::swzA(row)) << 4)) = v;
      else *TNX_LDS(i32x4, stage_base + C::A_BYTES + row * C::ROWB_B + ((cs ^ C::swzB(row)) << 4)) = v;
    }
  };
  auto gen_fetch = [&](int kt_global, int t0, i32x4 (&ra)[GEN_NA], i32x4 (&rb)[GEN_NB]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < GEN_NA; ++u) ra[u] = gen_fetch_a(kt_global, t0 + u * C::THREADS);
#pragma unroll
    for (int u = 0; u < GEN_NB; ++u) rb[u] = gen_fetch_b(kt_global, t0 + u * C::THREADS);
  };
  auto gen_store = [&](uint32_t stage_base, int t0, const i32x4 (&ra)[GEN_NA], const i32x4 (&rb)[GEN_NB]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < GEN_NA; ++u) gen_store_a(stage_base, t0 + u * C::THREADS, ra[u]);
#pragma unroll
    for (int u = 0; u < GEN_NB; ++u) gen_store_b(stage_base, t0 + u * C::THREADS, rb[u]);
  };
  // one chunk at a time: for the prologue of the kernels without the DMA loader, and for the left-out slab of operands whose rows are
  // shorter than a chunk or, with a row-major B, of at most one chunk of k
  auto load_slab_generic = [&](int kt_global, uint32_t stage_base, int t0) __attribute__((always_inline)) {
#pragma unroll 1
    for (int idx = t0; idx < BM * C::CPR_A; idx += C::THREADS) gen_store_a(stage_base, idx, gen_fetch_a(kt_global, idx));
#pragma unroll 1
    for (int idx = t0; idx < GEN_B_ROWS * GEN_B_CPR; idx += C::THREADS) gen_store_b(stage_base, idx, gen_fetch_b(kt_global, idx));
  };

  // The left-out slab of a tail_slab launch, with the DMA kernels' unit strides: all of a thread's chunks are on their way before the
  // first is waited for.  One chunk after another, each under conditions of its own, as load_slab_generic does it, cost a latency
  // apiece with nothing to hide it (447 x 14336 x 83 int8, BT: 11.7 -> 9.2 us; 256 x 872 x 904 8.2 -> 6.4; 1150 x 2300 x 1111 bf16 18.0 -> 17.1).
  // What lies past k is cleared; a chunk that crosses n, or m of an m-contiguous A, brings what comes after it, for columns that are never
  // stored.  Only in the matrix's last row is there nothing after it: such a chunk is fetched as the row's last 16 bytes and shifted
  // down.  That the other rows do have something after them is what the layouts' pitch >= length is for (dma_layout: loose_ok).  Rows
  // and chunks that do not exist read the first one's place.
  auto load_tail = [&](int kt_global, uint32_t stage_base, int t0) __attribute__((always_inline)) {
    const int64_t k0 = (int64_t)kt_global * BK;
    const int krem = (int)(p.k - k0);                               // 1 .. BK
    struct Side {
      const uint8_t* base;
      int64_t ld;
      int rows, left, odd;         // rows of the slab, elements of a row from the slab's first on, elements of a row past whole chunks
      bool ends;                   // a chunk that crosses the end of the matrix's last row
    };
    auto side = [&](const uint8_t* base, int64_t ld, int rows, bool last_row, int64_t left, int64_t len, int span) __attribute__((always_inline)) {
      const int odd = (int)(len % EPC);
      return Side{base, ld, rows, left < span ? (int)left : span, odd, last_row && odd != 0 && left < span};
    };
    auto fetch = [&](const Side& d, auto ntag, int cpr, int count, i32x4* r) __attribute__((always_inline)) {
      constexpr int N = decltype(ntag)::value;
#pragma unroll
      for (int u = 0; u < N; ++u) {
        int idx = t0 + u * C::THREADS;
        if (N * C::THREADS != count) idx = idx < count ? idx : count - 1;
        int row = idx / cpr, pos = idx % cpr * EPC;
        const bool none = row >= d.rows || pos >= d.left;
        row = none ? 0 : row;
        pos = none ? 0 : pos;
        pos = d.ends && row == d.rows - 1 && pos + EPC > d.left ? d.left - EPC : pos;
        r[u] = *(const gen_chunk_t*)(d.base + (uint32_t)((int64_t)row * d.ld * ES) + (int64_t)(pos * ES));
      }
      if (d.ends) {
        const int cut = (EPC - d.odd) * ES;                         // bytes a crossing chunk moves down
#pragma unroll
        for (int u = 0; u < N; ++u) {
          const int idx = t0 + u * C::THREADS, pos = idx % cpr * EPC;
          if (idx / cpr == d.rows - 1 && pos < d.left && pos + EPC > d.left) {
            uint32_t w[4] = {(uint32_t)r[u].x, (uint32_t)r[u].y, (uint32_t)r[u].z, (uint32_t)r[u].w};
#pragma unroll
            for (int by = 8; by >= 4; by /= 2) {
#pragma unroll
              for (int i = 0; i < 4; ++i) w[i] = cut & by ? (i + by / 4 < 4 ? w[i + by / 4] : 0u) : w[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = (uint32_t)(((uint64_t)(i < 3 ? w[i + 1] : 0u) << 32 | w[i]) >> ((cut & 3) * 8));
            r[u] = i32x4{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
          }
        }
      }
    };
    // k along the row: elements past k; k rows: rows past k
    auto clear_k = [&](const Side& d, auto ntag, int cpr, i32x4* r) __attribute__((always_inline)) {
      constexpr int N = decltype(ntag)::value;
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int valid = (d.left - (t0 + u * C::THREADS) % cpr * EPC) * ES;      // bytes
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int bytes = valid - 4 * i;
          r[u][i] &= bytes >= 4 ? -1 : bytes <= 0 ? 0 : (1 << bytes * 8) - 1;
        }
      }
    };
    auto clear_rows = [&](auto ntag, int cpr, i32x4* r) __attribute__((always_inline)) {
      constexpr int N = decltype(ntag)::value;
#pragma unroll
      for (int u = 0; u < N; ++u)
        if ((t0 + u * C::THREADS) / cpr >= krem) r[u] = i32x4{0, 0, 0, 0};
    };
    const int64_t len_a = AT ? p.m : p.k, len_b = BT ? p.k : p.n;
    // (a row-major B and one chunk of k: what exists is a few rows of B and one chunk of each row of A, and the loop that skips
    // the rest takes no longer -- 1025 x 2050 x 4100 36.1 us against 36.6, 1100 x 1100 x 1027 11.2 against 11.5)
    if (len_a < EPC || len_b < EPC || (!BT && krem <= EPC)) {
      load_slab_generic(kt_global, stage_base, t0);
      return;
    }
    constexpr int CPR_A = AT ? AT_CPR : C::CPR_A;
    const int64_t lda = AT ? p.sak : p.sam, ldb = BT ? p.sbn : p.sbk, mleft = p.m - m0, nleft = p.n - n0;
    const Side da = AT ? side(p.a + (k0 * lda + m0) * ES, lda, krem, true, mleft, len_a, BM)
                       : side(p.a + (m0 * lda + k0) * ES, lda, mleft < BM ? (int)mleft : BM, mleft <= BM, krem, len_a, BK);
    const Side db = BT ? side(p.b + (n0 * ldb + k0) * ES, ldb, nleft < BN ? (int)nleft : BN, nleft <= BN, krem, len_b, BK)
                       : side(p.b + (k0 * ldb + n0) * ES, ldb, krem, true, nleft, len_b, BN);
    i32x4 ra[GEN_NA], rb[GEN_NB];
    fetch(da, IntTag<GEN_NA>{}, CPR_A, BM * C::CPR_A, ra);
    fetch(db, IntTag<GEN_NB>{}, GEN_B_CPR, GEN_B_ROWS * GEN_B_CPR, rb);
    if constexpr (AT) clear_rows(IntTag<GEN_NA>{}, CPR_A, ra);
    else clear_k(da, IntTag<GEN_NA>{}, CPR_A, ra);
    if constexpr (BT) clear_k(db, IntTag<GEN_NB>{}, GEN_B_CPR, rb);
    else clear_rows(IntTag<GEN_NB>{}, GEN_B_CPR, rb);
    gen_store(stage_base, t0, ra, rb);
  };

  // CONV: the first 64 threads write the taps of the next slab to tabulate into the table of its parity and move
  // their tap one slab on; every lane reads the entries of its ops of the slab that is about to be issued.
  auto conv_tab_write = [&]() __attribute__((always_inline)) {
    if constexpr (CONV) {
      const ConvGeom& g = p.cv;
      if (wave == 0) {
        *TNX_LDS(i32x2, cv_ktab + (uint32_t)(cv_wr & 1) * (BK * 8) + (uint32_t)lane * 8u) =
            i32x2{(int)tap_off, (int)((uint32_t)tap_dh | ((uint32_t)tap_dw << 16))};
        int ndw = tap_dw + g.step_dw;
        const bool wrap_w = ndw >= g.lim_w;
        ndw -= wrap_w ? g.lim_w : 0;
        int ndh = tap_dh + g.step_dh + (wrap_w ? g.dil_h : 0);
        const bool wrap_h = ndh >= g.lim_h;
        ndh -= wrap_h ? g.lim_h : 0;
        tap_off += (uint32_t)(g.step_koff + (wrap_w ? g.adj_w : 0) + (wrap_h ? g.adj_h : 0));
        tap_dw = ndw;
        tap_dh = ndh;
      }
      ++cv_wr;
    }
  };
  auto conv_tab_read = [&]() __attribute__((always_inline)) {
    if constexpr (CONV) {
#pragma unroll
      for (int qb = 0; qb < C::B_LPW; ++qb)
        cv_ent[qb] = *TNX_LDS(i32x2, cv_ktab + (uint32_t)(cv_rd & 1) * (BK * 8) + (uint32_t)(qb * CONV_STEP + cv_r0) * 8u);
      ++cv_rd;
    }
  };
  // CONV: byte offset of B op qb's chunk inside the input (or CV_OUTSIDE) and its fix-up note
  uint32_t cv_voff = 0;
  auto conv_prepare = [&](int qb, uint32_t stage_base) __attribute__((always_inline)) {
    const ConvGeom& g = p.cv;
    const int row = qb * CONV_STEP + cv_r0;
    const bool second = ((row >> 3) ^ (row >> 4)) & 1;      // the pass term of swzB
    const int off = second ? pix_off1 : pix_off0, hw = second ? pix_hw1 : pix_hw0;
    const int h0 = hw >> 16, w0 = (int)(int16_t)(hw & 0xffff);
    const int dh = cv_ent[qb].y & 0xffff, dw = (int)((uint32_t)cv_ent[qb].y >> 16);
    const int o = off + cv_ent[qb].x;
    int lo = -(w0 + dw), hi = g.w_in - (w0 + dw);            // elements [lo, hi) of the chunk lie inside the input row
    lo = lo < 0 ? 0 : lo;
    hi = hi > 8 ? 8 : hi;
    const bool ok = (uint32_t)(h0 + dh) < (uint32_t)g.h_in && lo < hi;
    // A chunk that starts before the tensor (first row of the first image, left padding) or ends after it (last
    // row of the last image, right padding) cannot be fetched whole: the buffer bound drops every dword that is not
    // entirely inside, valid elements included (a negative offset wraps to one past every bound).  Its inside
    // elements are written by the fix-up, which recognises the case from the offset kept here.
    cv_voff = ok ? (uint32_t)o * 2u : CV_OUTSIDE;
    cv_fix[qb] = ok ? (uint32_t)(lo * 9 + hi) * 16u : CV_NOFIX;
    cv_o[qb] = o;
    cv_dst = stage_base;
    cv_pending = true;
  };
  auto conv_go = [&]() __attribute__((always_inline)) {
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(cv_voff), "s"(cv_rsrc) : "memory");
  };
  // Fix-up of one op's chunk: zero the elements outside [lo, hi): chunk & mask(lo, hi), the mask read from the
  // table.  In two parts so that the two LDS reads have returned when the second part runs: fix_read, a few MFMA
  // slots, fix_write.  Every lane does it for every op, needed or not (its mask is all ones when it has nothing to
  // zero): straight-line code lets the compiler wait for exactly these reads, where a branch around them made it
  // wait for every LDS read in flight (measured: 433 with the branch, 618 TFLOP/s with no fix-up at all).
  // A chunk that could not be fetched whole at either end of the tensor (conv_prepare) was loaded as zeros and
  // has its inside elements filled in one by one afterwards (fix_special); that happens in a handful of
  // workgroups at most and costs the others one uniform branch per period.
  i32x4 cv_rmw[CONV ? C::B_LPW : 1], cv_msk[CONV ? C::B_LPW : 1];
  auto conv_fix_at = [&](int qb, uint32_t dst) __attribute__((always_inline)) {
    return dst + C::A_BYTES + (uint32_t)(qb * NW + wave) * 1024u + (uint32_t)lane * 16u;
  };
  auto conv_fix_read = [&](int qb, uint32_t note, uint32_t dst) __attribute__((always_inline)) {
    cv_msk[qb] = *TNX_LDS(i32x4, cv_table + (note & 0xffffu));
    cv_rmw[qb] = *TNX_LDS(i32x4, conv_fix_at(qb, dst));
  };
  auto conv_fix_write = [&](int qb, uint32_t note, uint32_t dst) __attribute__((always_inline)) {
    *TNX_LDS(i32x4, conv_fix_at(qb, dst)) = cv_rmw[qb] & cv_msk[qb];
  };
  auto conv_fix_special = [&](const uint32_t (&notes)[CONV ? C::B_LPW : 1], const int (&os)[CONV ? C::B_LPW : 1],
                              uint32_t dst) __attribute__((always_inline)) {
    const int x_elems = (int)(p.cv.x_bytes >> 1);
    bool any = false;
#pragma unroll
    for (int qb = 0; qb < (CONV ? C::B_LPW : 0); ++qb) any |= notes[qb] != CV_NOFIX && (os[qb] < 0 || os[qb] > x_elems - 8);
    if (__builtin_amdgcn_ballot_w64(any) != 0) {
#pragma unroll 1
      for (int qb = 0; qb < (CONV ? C::B_LPW : 0); ++qb) {
        uint32_t note = CV_NOFIX;
        int o = 0;
#pragma unroll
        for (int x = 0; x < (CONV ? C::B_LPW : 0); ++x) {   // no register-indexed array
          note = x == qb ? notes[x] : note;
          o = x == qb ? os[x] : o;
        }
        if (note != CV_NOFIX && (o < 0 || o > x_elems - 8)) {
          const uint32_t at = conv_fix_at(qb, dst);
          const int idx = (int)(note >> 4), lo = idx / 9, hi = idx % 9;
          const uint16_t* src = (const uint16_t*)p.b + o;
#pragma unroll 1
          for (int e = lo; e < hi; ++e) *TNX_LDS(uint16_t, at + 2 * e) = src[e];
        }
      }
    }
  };
  // the whole fix-up of the slab whose notes are in `notes`, in one go (prologue and the first draining period)
  auto conv_fixup_all = [&](const uint32_t (&notes)[CONV ? C::B_LPW : 1], const int (&os)[CONV ? C::B_LPW : 1],
                            uint32_t dst) __attribute__((always_inline)) {
    if constexpr (CONV) {
#pragma unroll
      for (int qb = 0; qb < C::B_LPW; ++qb) conv_fix_read(qb, notes[qb], dst);
#pragma unroll
      for (int qb = 0; qb < C::B_LPW; ++qb) conv_fix_write(qb, notes[qb], dst);
      conv_fix_special(notes, os, dst);
    }
  };
  auto conv_fixup = [&]() __attribute__((always_inline)) {
    if constexpr (CONV) {
      if (cv_pending) {
        conv_fixup_all(cv_fix, cv_o, cv_dst);
        cv_pending = false;
      }
    }
  };
  // Inside a period the fix-up works on a copy of the notes taken when the period starts (the period's own B ops
  // write new notes): part one of op qb behind MFMA slot CV_FS * qb, part two CV_FD slots later.
  uint32_t cv_old[CONV ? C::B_LPW : 1];
  int cv_old_o[CONV ? C::B_LPW : 1];
  uint32_t cv_old_dst = 0;
  // ... and the lanes fetch the table entries of the slab this period issues, and the first 64 threads tabulate the
  // slab after it (into the table that was last read one period ago, before the barrier that has just been passed)
  auto conv_period_begin = [&]() __attribute__((always_inline)) {
    if constexpr (CONV) {
#pragma unroll
      for (int qb = 0; qb < C::B_LPW; ++qb) { cv_old[qb] = cv_fix[qb]; cv_old_o[qb] = cv_o[qb]; }
      cv_old_dst = cv_dst;
      conv_tab_read();
      conv_tab_write();
    }
  };
  // The period's own loads are all issued in its first half; in the middle of the period the wave waits until only
  // those are outstanding, i.e. until the slab issued one period earlier has landed (loads retire in issue order),
  // and fixes that slab in the second half.  A slab so has a period and a half to arrive.
  constexpr int CV_PERIOD = C::KSTEPS * TM * TN;
  constexpr int CV_WAIT_SLOT = CV_PERIOD / 2;
  constexpr int CV_FD = CV_PERIOD >= 32 ? 6 : 3;                                        // slots between read and write
  constexpr int CV_FS = !CONV ? 1 : ((CV_PERIOD / 2 - CV_FD - 3) / C::B_LPW >= 4 ? 4 : ((CV_PERIOD / 2 - CV_FD - 3) / C::B_LPW >= 2 ? 2 : 1));
  static_assert(!CONV || CV_WAIT_SLOT + 1 + CV_FS * (C::B_LPW - 1) + CV_FD + 1 < CV_PERIOD, "no room for the fix-up in half a period");
  auto conv_fix_slot = [&](int slot) __attribute__((always_inline)) {
    if constexpr (CONV) {
      if (slot == CV_WAIT_SLOT) { TNX_WAIT_VM(C::LPW); }
#pragma unroll
      for (int qb = 0; qb < C::B_LPW; ++qb) {
        if (slot == CV_WAIT_SLOT + 1 + CV_FS * qb) conv_fix_read(qb, cv_old[qb], cv_old_dst);
        if (slot == CV_WAIT_SLOT + 1 + CV_FS * qb + CV_FD) conv_fix_write(qb, cv_old[qb], cv_old_dst);
      }
      if (slot == CV_WAIT_SLOT + 1 + CV_FS * (C::B_LPW - 1) + CV_FD + 1) conv_fix_special(cv_old, cv_old_o, cv_old_dst);
    }
  };

  auto gather_go = [&](int qb) __attribute__((always_inline)) {
    asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" : : "v"(b_voff[qb] + g_tap), "s"(g_rsrc) : "memory");
  };
  auto gather_next = [&]() __attribute__((always_inline)) {
    if constexpr (GATHER) {
      g_tap = *TNX_LDS(uint32_t, g_at);
      g_at += g_whole ? 4 : 32;
    }
  };

  // one DMA op (q-th of this wave) of local slab t, into ring slot t % STAGES
  auto dma_op = [&](int q, uint32_t stage_base) __attribute__((always_inline)) {
    if (CONV && q >= C::A_LPW) {
      conv_prepare(q - C::A_LPW, stage_base);
      dma16_set_m0(stage_base + C::A_BYTES + ((q - C::A_LPW) * NW + wave) * 1024);
      asm volatile("s_nop 0" ::: "memory");
      conv_go();
    } else if (q < C::A_LPW) {
      dma16(a_sbase, a_voff[q], stage_base + (q * NW + wave) * 1024);
    } else if (GATHER) {
      dma16_set_m0(stage_base + C::A_BYTES + b_op(q - C::A_LPW) * 1024);
      asm volatile("s_nop 0" ::: "memory");
      gather_go(q - C::A_LPW);
    } else {
      // short tiles are the ones used on skinny problems, where B is the HBM stream
      if (BM <= 64 && p.b_once)
        dma16_nt(b_sbase, b_voff[q - C::A_LPW], stage_base + C::A_BYTES + ((q - C::A_LPW) * NW + wave) * 1024);
      else
        dma16(b_sbase, b_voff[q - C::A_LPW], stage_base + C::A_BYTES + ((q - C::A_LPW) * NW + wave) * 1024);
    }
  };
  // the same op in two parts (see dma16_set_m0): LDS target first, the load after one other instruction
  auto dma_target = [&](int q, uint32_t stage_base) __attribute__((always_inline)) {
    if (CONV && q >= C::A_LPW) conv_prepare(q - C::A_LPW, stage_base);
    if (q < C::A_LPW) dma16_set_m0(stage_base + (q * NW + wave) * 1024);
    else dma16_set_m0(stage_base + C::A_BYTES + b_op(q - C::A_LPW) * 1024);
  };
  auto dma_go = [&](int q) __attribute__((always_inline)) {
    if (CONV && q >= C::A_LPW) conv_go();
    else if (GATHER && q >= C::A_LPW) gather_go(q - C::A_LPW);
    else if (q < C::A_LPW) dma16_go<false>(a_sbase, a_voff[q]);
    else if (BM <= 64 && p.b_once) dma16_go<true>(b_sbase, b_voff[q - C::A_LPW]);
    else dma16_go<false>(b_sbase, b_voff[q - C::A_LPW]);
  };
  auto dma_advance = [&]() __attribute__((always_inline)) {
    if (TNX_LADDER == 3) return;        // + DMA ops, always of the tile's first slabs (served by the L2)
    a_sbase += AT ? (int64_t)BK * p.sak * ES : (int64_t)BK * ES;
    if (GATHER) gather_next();
    else if (!CONV) b_sbase += BT ? (int64_t)BK * ES : (int64_t)BK * p.sbk * ES;
  };
  auto stage_of = [&](int t) __attribute__((always_inline)) { return lds0 + (uint32_t)(t % STAGES) * C::STAGE_BYTES; };

  // ---- fragment addressing ----------------------------------------------
  const int wy = wave / C::WGN, wx = wave % C::WGN;
  const int a_row = wy * C::WTM + (lane % MI);
  const int a_kg = lane / MI;
  const int a_sw = C::swzA(a_row);
  uint32_t a_koff[C::KSTEPS];   // byte offset inside the A slab, per k step
#pragma unroll
  for (int ks = 0; ks < C::KSTEPS; ++ks)
    a_koff[ks] = a_row * C::ROWB_A + (((ks * (C::KB / 16) + a_kg) ^ a_sw) << 4);

  const int blk = lane >> 4, li = lane & 15;
  const int b_kg = (MI == 32) ? (blk >> 1) : blk;
  const int b_sub = (ES == 4) ? 0 : (ES == 2) ? (li >> 2) : (li >> 1);               // k row inside the transposed block
  const int b_col = (ES == 4) ? 4 * li : (ES == 2) ? 8 * (li & 3) : 8 * (li & 1);    // byte of the block's row
  const int b_colb0 = (wx * C::WTN + ((MI == 32) ? 16 * (blk & 1) : 0)) * ES + b_col;
  constexpr int RPR = 8 / ES;                                       // k rows one transposing read covers
  const int b_sw = C::swzB((16 / ES) * b_kg + b_sub);     // the same for every k step and both halves of a fragment
  uint32_t b_joff[TN];          // byte offset inside the B slab, per column block
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    int colb = b_colb0 + j * MI * ES;
    b_joff[j] = (uint32_t)(((16 / ES) * b_kg + b_sub) * C::ROWB_B) + (((colb >> 4) ^ b_sw) << 4) + (colb & 15);
  }

  // m-contiguous A: as a row-major B slab
  const int at_colb0 = (wy * C::WTM) * ES + b_col;
  const int at_sw = C::template swzT<AT_CPR>((16 / ES) * b_kg + b_sub);
  uint32_t at_off[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    int colb = at_colb0 + i * MI * ES;
    at_off[i] = (uint32_t)(((16 / ES) * b_kg + b_sub) * AT_ROWB) + (((colb >> 4) ^ at_sw) << 4) + (colb & 15);
  }

  // k-contiguous B: fragment j of k step ks sits at bt_koff[ks] + j * MI rows, read like an A fragment
  const int bt_row = wx * C::WTN + (lane % MI);
  uint32_t bt_koff[C::KSTEPS];
#pragma unroll
  for (int ks = 0; ks < C::KSTEPS; ++ks)
    bt_koff[ks] = bt_row * C::ROWB_A + (((ks * (C::KB / 16) + a_kg) ^ C::swzA(bt_row)) << 4);

  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{};

  // two register sets of fragments: one being multiplied, one being filled
  i32x4 fa[2][TM];
  i32x2 fb[2][TN][2];
  i32x2 fat[2][TM][2];          // m-contiguous A: two transposing reads per fragment
  i32x4 fbq[2][TN];             // k-contiguous B: one 16-byte read per fragment
  constexpr int NBREAD = BT ? TN : 2 * TN;
  constexpr int NREAD = NBREAD + (AT ? 2 * TM : TM), NMMA = TM * TN;
  constexpr int RPM = (NREAD + NMMA - 1) / NMMA;        // LDS reads slotted behind each MFMA
  constexpr int DPM = (C::LPW + NMMA - 1) / NMMA;       // DMA ops slotted behind each MFMA

  // The swizzle XORs chunk-index bits that hold nothing but the fragment's number, so the offset of fragment j of an A^T
  // or B slab is that of fragment 0 with j * MI * ES XOR-ed in.  The 256-wide AT tiles form it that way, one vector
  // instruction per fragment: kept in registers, 12 offsets for each of two slots (which lie further apart than an LDS
  // instruction's immediate reaches) spill inside the K loop (4096 x 4096 x 2048: 184 us, with the XOR 55).  The asm
  // keeps the compiler from computing them ahead of the loop all the same.
  constexpr bool XOR_OFFS = AT && C::STAGE_BYTES >= 65536;
  uint32_t xo_at = 0, xo_b = 0;
  auto xor_off = [&](uint32_t base, int bits) __attribute__((always_inline)) {
    uint32_t r;
    asm volatile("v_xor_b32 %0, %1, %2" : "=v"(r) : "i"(bits), "v"(base));
    return r;
  };
  // Likewise the 256-wide float32 pairs of a k-contiguous B: an offset for each operand, k step and slot, kept in registers, takes
  // eight where the loop has two to spare (packed conv2d: 96 registers spilled, 21 reloads per two slabs; now one).  The k step is
  // again a bit to XOR in, the slot is added in the same instruction.
  constexpr bool SLOT_OFFS = BT && PAIR && C::STAGE_BYTES >= 65536;
  static_assert(!SLOT_OFFS || (MI == 16 && C::BK * ES == 128), "the k step is one bit of the chunk index");
  uint32_t so_a = 0, so_b = 0;
  auto slot_off = [&](uint32_t slot, uint32_t off, int ks) __attribute__((always_inline)) {
    uint32_t r;
    asm volatile("v_xad_u32 %0, %1, %2, %3" : "=v"(r) : "v"(off), "i"(ks * C::KB), "s"(slot));
    return r;
  };
  auto read_one = [&](int set, int idx, uint32_t sa, uint32_t sb, int ks) __attribute__((always_inline)) {
    if (BT && idx < NBREAD) {
      if constexpr (SLOT_OFFS) {
        if (idx == 0) so_b = slot_off(sb, bt_koff[0], ks);
        fbq[set][idx] = *TNX_LDS(i32x4, so_b + idx * MI * C::ROWB_A);
      } else {
        fbq[set][idx] = *TNX_LDS(i32x4, sb + bt_koff[ks] + idx * MI * C::ROWB_A);
      }
    } else if (idx < NBREAD) {
      int j = idx >> 1, h = idx & 1;
      if constexpr (XOR_OFFS) {
        if (h == 0) xo_b = xor_off(sb + b_joff[0], j * MI * ES);
        fb[set][j][h] = lds_read_tr<ES, C::ROWB_B>(xo_b + ks * C::MMA_K * C::ROWB_B + h * RPR * C::ROWB_B);
      } else {
        fb[set][j][h] = lds_read_tr<ES, C::ROWB_B>(sb + b_joff[j] + ks * C::MMA_K * C::ROWB_B + h * RPR * C::ROWB_B);
      }
    } else if (AT) {
      int i = (idx - NBREAD) >> 1, h = (idx - NBREAD) & 1;
      if constexpr (XOR_OFFS) {
        if (h == 0) xo_at = xor_off(sa + at_off[0], i * MI * ES);
        fat[set][i][h] = lds_read_tr<ES, AT_ROWB>(xo_at + ks * C::MMA_K * AT_ROWB + h * RPR * AT_ROWB);
      } else {
        fat[set][i][h] = lds_read_tr<ES, AT_ROWB>(sa + at_off[i] + ks * C::MMA_K * AT_ROWB + h * RPR * AT_ROWB);
      }
    } else {
      int i = idx - NBREAD;
      if constexpr (SLOT_OFFS) {
        if (i == 0) so_a = slot_off(sa, a_koff[0], ks);
        fa[set][i] = *TNX_LDS(i32x4, so_a + i * MI * C::ROWB_A);
      } else {
        fa[set][i] = *TNX_LDS(i32x4, sa + a_koff[ks] + i * MI * C::ROWB_A);
      }
    }
  };
  auto mma_at = [&](int set_a, int set_b, int i, int j) __attribute__((always_inline)) {
    i32x4 b4 = BT ? fbq[set_b][j] : i32x4{fb[set_b][j][0].x, fb[set_b][j][0].y, fb[set_b][j][1].x, fb[set_b][j][1].y};
    i32x4 a4 = AT ? i32x4{fat[set_a][i][0].x, fat[set_a][i][0].y, fat[set_a][i][1].x, fat[set_a][i][1].y} : fa[set_a][i];
    acc[i][j] = MMA::run(b4, a4, acc[i][j]);   // rows = n, cols = m: the tile comes out transposed
  };
  auto mma_one = [&](int set, int idx) __attribute__((always_inline)) {
    int i = idx / TN, j = idx % TN;
    if (i & 1) j = TN - 1 - j;   // serpentine walk of the wave's MFMA tiles: one operand changes per instruction, never both
    mma_at(set, set, i, j);
  };

  // ---- pipeline ----------------------------------------------------------
  // Ring of STAGES slabs, one workgroup barrier per slab.  barrier(t) sits
  // before the last k step of slab t: every wave has then issued and received
  // all its LDS reads of slab t, so the slot of slab t is handed to the DMA of
  // slab t+STAGES, and slab t+1 is known to have landed, so its first
  // fragments are fetched under the last k step's MFMAs.  A "period" is the
  // code between barrier(t) and barrier(t+1): the last k step of slab t, then
  // k steps 0..KSTEPS-2 of slab t+1.  The DMA ops of one refill are slotted
  // behind the period's MFMAs at an even rate (a burst of them backs up the
  // texture-address queue and stalls the wave); with only two slabs in the
  // ring the refill is due at the very next barrier, so it is issued in the
  // first k step of the period instead.  The K loop is cut in three (refills
  // to issue / ring draining / final step) so the accumulators flow through
  // straight-line code.
  constexpr int PERIOD = (PAIR ? 3 : C::KSTEPS) * NMMA;            // MFMA slots per period
  // slots the refill is spread over.  Two-slab rings: the refill is due at the next barrier, so it
  // is front-loaded: over the first half of the period with one wave per SIMD (measured on 8192^3,
  // bf16 256x256x64: a quarter of the period 477, three eighths 853, half 1430, three quarters
  // 1380 TFLOP/s -- a faster burst backs up the texture address path and stalls the wave for far
  // longer than it saves; spread further, the last loads are waited for as soon as they are
  // issued), over the first quarter with two waves per SIMD (the other wave covers the stall).
  constexpr int SPAN2 = (NW == 4 ? PERIOD / 2 : PERIOD / 4) > 0 ? (NW == 4 ? PERIOD / 2 : PERIOD / 4) : 1;
  // (CONV: three slots, but every load is waited for at the next barrier as with two)
  constexpr int SPAN = (STAGES == 2 || !FAST || CONV) ? SPAN2 : PERIOD;
  // loads of this wave that may still be in flight when a period starts (CONV: the slab issued in the period
  // before, which is waited for in the middle of this one)
  constexpr int PWAIT = CONV ? C::LPW : (STAGES - 2) * C::LPW;
  constexpr int LAST = (C::KSTEPS - 1) & 1;                      // register set holding the last k step
  constexpr int NEXT0 = C::KSTEPS & 1;                           // set that receives step 0 of the next slab

  // One MFMA slot: the MFMA, then the LDS reads and DMA ops slotted behind it.  When exactly one DMA op and at
  // least one read are due, the read sits between the op's M0 write and its load (it fills the wait state).
  auto slot_body = [&](int mset, int x, int rset, int& rd, uint32_t sa, uint32_t sb, int ks_next, bool with_dma, int slot,
                       uint32_t dst) __attribute__((always_inline)) {
    mma_one(mset, x);
    if (TNX_LADDER == 1) {              // MFMAs only
      __builtin_amdgcn_sched_barrier(0);
      return;
    }
    if (TNX_LADDER == 2) with_dma = false;   // + fragment reads: the ring keeps the slabs of the prologue
    if (with_dma) conv_fix_slot(slot);
    int lo = 0, hi = 0;
    if (with_dma && slot < SPAN) { lo = slot * C::LPW / SPAN; hi = (slot + 1) * C::LPW / SPAN; }
    const bool paired = hi - lo == 1 && rd < NREAD;
    if (paired) dma_target(lo, dst);
#pragma unroll
    for (int q = 0; q < RPM; ++q)
      if (rd < NREAD) { read_one(rset, rd, sa, sb, ks_next); ++rd; }
    if (paired) dma_go(lo);
    else
#pragma unroll
      for (int q = lo; q < hi; ++q) dma_op(q, dst);
    __builtin_amdgcn_sched_barrier(0);
  };
  // `par` (0 or 1, compile-time) is added to every register-set index: with an odd number of k steps per slab
  // the two sets trade roles from one slab to the next, and the unrolled bulk of the K loop follows that by
  // alternating par; where the slab index is a run-time value (par = 0) the sets are swapped by copying.
  auto inner_steps = [&](uint32_t sa, uint32_t sb, auto with_dma, uint32_t dst, auto par) __attribute__((always_inline)) {
    constexpr bool WITH_DMA = decltype(with_dma)::value;
    constexpr int P = decltype(par)::value;
#pragma unroll
    for (int ks = 0; ks + 1 < C::KSTEPS; ++ks) {
      int rd = 0;
#pragma unroll
      for (int x = 0; x < NMMA; ++x)
        slot_body((ks + P) & 1, x, (ks + 1 + P) & 1, rd, sa, sb, ks + 1, WITH_DMA, (PAIR ? 2 : 1) * NMMA + ks * NMMA + x, dst);
    }
  };
  // last k step of the slab whose fragments sit in set LAST; prefetches step 0 of the slab at (sa1, sb1)
  // (`par` is the parity of the slab that is ending; `swap`: bring the sets back to par = 0 by copying)
  auto last_step = [&](uint32_t sa1, uint32_t sb1, auto with_dma, uint32_t dst, auto par, auto swap) __attribute__((always_inline)) {
    constexpr bool WITH_DMA = decltype(with_dma)::value;
    constexpr int P = decltype(par)::value;
    int rd = 0;
#pragma unroll
    for (int x = 0; x < NMMA; ++x) slot_body((LAST + P) & 1, x, (NEXT0 + P) & 1, rd, sa1, sb1, 0, WITH_DMA, x, dst);
    if ((C::KSTEPS & 1) && decltype(swap)::value) {   // odd KSTEPS: the two register sets trade roles every slab
#pragma unroll
      for (int i = 0; i < TM; ++i) { i32x4 tmp = fa[0][i]; fa[0][i] = fa[1][i]; fa[1][i] = tmp; }
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) { i32x2 tmp = fb[0][j][h]; fb[0][j][h] = fb[1][j][h]; fb[1][j][h] = tmp; }
#pragma unroll
      for (int j = 0; j < TN; ++j) { i32x4 tmp = fbq[0][j]; fbq[0][j] = fbq[1][j]; fbq[1][j] = tmp; }
    }
  };
  typedef BoolTag<true> Yes;
  typedef BoolTag<false> No;
  typedef IntTag<0> Par0;
  // PAIR: what takes the place of the last k step.  Heads are in set 0, already multiplied with each other; the tails
  // of the same 32 k have arrived in set 1.  First A's tails with B's heads column by column, then A's heads with B's
  // tails row by row: so set 0 falls free one fragment after another, B's first, and the next slab's heads are read
  // into it behind the MFMAs without a third set of registers (which the 256-wide tiles do not have).
  auto cross_step = [&](uint32_t sa1, uint32_t sb1, auto with_reads, auto with_dma, uint32_t dst) __attribute__((always_inline)) {
    constexpr bool READS = decltype(with_reads)::value, WITH_DMA = decltype(with_dma)::value;
    constexpr int RB = BT ? 1 : 2, RA = AT ? 2 : 1;
    auto read_b = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < RB; ++h) read_one(0, j * RB + h, sa1, sb1, 0);
    };
    auto read_a = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < RA; ++h) read_one(0, NBREAD + i * RA + h, sa1, sb1, 0);
    };
#pragma unroll
    for (int s = 0; s < 2 * NMMA; ++s) {
      if (s < NMMA) {
        const int j = s / TM, i = s % TM;
        mma_at(1, 0, (j & 1) ? TM - 1 - i : i, j);
      } else {
        const int i = (s - NMMA) / TN, j = (s - NMMA) % TN;
        mma_at(0, 1, i, (i & 1) ? TN - 1 - j : j);
      }
      int lo = 0, hi = 0;
      if (WITH_DMA && s < SPAN) { lo = s * C::LPW / SPAN; hi = (s + 1) * C::LPW / SPAN; }
      const bool rb = READS && s >= TM && s <= NMMA && s % TM == 0, ra = READS && s > NMMA && (s - NMMA) % TN == 0;
      const bool paired = hi - lo == 1 && (rb || ra);
      if (paired) dma_target(lo, dst);
      if (rb) read_b(s / TM - 1);
      if (ra) read_a((s - NMMA) / TN - 1);
      if (paired) dma_go(lo);
      else
#pragma unroll
        for (int q = lo; q < hi; ++q) dma_op(q, dst);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (READS) read_a(TM - 1);
  };
  // what follows a barrier: the end of the slab whose fragments are in registers
  auto end_slab = [&](uint32_t sa1, uint32_t sb1, auto with_dma, uint32_t dst, auto par, auto swap) __attribute__((always_inline)) {
    if constexpr (PAIR) cross_step(sa1, sb1, Yes{}, with_dma, dst);
    else last_step(sa1, sb1, with_dma, dst, par, swap);
  };

  // first STAGES slabs of the tile the loader stands on
  auto issue_prologue = [&]() __attribute__((always_inline)) {
    if constexpr (CONV) {
      // slabs 0 and 1 are read before any period could fix them: both are issued, waited for and fixed here;
      // slab 2 is issued afterwards and takes the regular route.  The tap tables of slabs 0..3 are written on the
      // way, each behind a barrier that separates it from the reads of the table it replaces; the table of slab 3
      // is published by the first period's barrier.
      uint32_t first[C::B_LPW];
      int first_o[C::B_LPW];
      const uint32_t dst0 = stage_of(0);
      conv_tab_write();                       // slab 0 -> table 0
      __syncthreads();
      conv_tab_read();
      if (KT > 0) {
#pragma unroll
        for (int q = 0; q < C::LPW; ++q) dma_op(q, dst0);
        dma_advance();
#pragma unroll
        for (int qb = 0; qb < C::B_LPW; ++qb) { first[qb] = cv_fix[qb]; first_o[qb] = cv_o[qb]; }
      }
      conv_tab_write();                       // slab 1 -> table 1
      __syncthreads();
      conv_tab_read();
      if (KT > 1) {
#pragma unroll
        for (int q = 0; q < C::LPW; ++q) dma_op(q, stage_of(1));
        dma_advance();
      }
      TNX_WAIT_VM(0);
      if (KT > 0) conv_fixup_all(first, first_o, dst0);
      if (KT > 1) conv_fixup_all(cv_fix, cv_o, stage_of(1));
      cv_pending = false;
      conv_tab_write();                       // slab 2 -> table 0 (its readers passed the barrier above)
      __syncthreads();
      conv_tab_read();
      if (KT > 2) {
#pragma unroll
        for (int q = 0; q < C::LPW; ++q) dma_op(q, stage_of(2));
        dma_advance();
      }
      conv_tab_write();                       // slab 3 -> table 1
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the fix-up writes are done before the barrier that follows
      return;
    }
    if constexpr (GATHER) {
      __syncthreads();                                  // the offset table is complete
      gather_next();
    }
#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
      if (s < KT) {
        if constexpr (FAST) {
#pragma unroll
          for (int q = 0; q < C::LPW; ++q) dma_op(q, stage_of(s));
          dma_advance();
        } else {
          load_slab_generic(kt0 + s, stage_of(s), tid);
        }
      }
    }
  };
  // the K loop of one tile, from "slab 0 has landed" to the last MFMA; the prologue has been issued
  auto k_loop = [&]() __attribute__((always_inline)) {
  if (KT > 0) {
    __syncthreads();
    const uint32_t sa = stage_of(0), sb = sa + C::A_BYTES;
#pragma unroll
    for (int r = 0; r < NREAD; ++r) read_one(0, r, sa, sb, 0);
    if (TNX_LADDER == 1) {
#pragma unroll
      for (int r = 0; r < NREAD; ++r) read_one(1, r, sa, sb, C::KSTEPS > 1 ? 1 : 0);
    }
    inner_steps(sa, sb, No{}, 0u, Par0{});
  }

  int t = 0;
  // (1) periods that issue the refill of slab t+STAGES into the slot of slab t.  The bulk runs
  // STAGES periods per trip so every ring slot is a compile-time constant there (LDS addresses
  // become instruction immediates, DMA targets become scalar constants); what is left over runs
  // with run-time slots.
  // With an odd number of k steps per slab the trip covers an even number of periods, so that the register
  // sets are back in their starting roles at the end of every trip without a copy.
  if constexpr (FAST) {
    constexpr int U = ((C::KSTEPS & 1) && (STAGES & 1)) ? 2 * STAGES : STAGES;
    for (; t + U + STAGES - 1 < KT; t += U) {
      auto period = [&](auto jtag) __attribute__((always_inline)) {
        constexpr int j = decltype(jtag)::value;
        constexpr int P = (C::KSTEPS & 1) ? (j & 1) : 0;          // parity of the slab whose last k step runs now
        if (TNX_LADDER != 1) {
          if (TNX_LADDER != 4) __builtin_amdgcn_s_waitcnt((PWAIT & 0xF) | (((PWAIT >> 4) & 0x3) << 14) | 0x0070);
          __builtin_amdgcn_s_barrier();
        }
        __builtin_amdgcn_sched_barrier(0);
        conv_period_begin();
        const uint32_t dst = lds0 + (uint32_t)(j % STAGES) * C::STAGE_BYTES;
        const uint32_t sa1 = lds0 + (uint32_t)((j + 1) % STAGES) * C::STAGE_BYTES, sb1 = sa1 + C::A_BYTES;
        end_slab(sa1, sb1, Yes{}, dst, IntTag<P>{}, No{});
        inner_steps(sa1, sb1, Yes{}, dst, IntTag<(C::KSTEPS & 1) ? (P ^ 1) : 0>{});
        dma_advance();
      };
      static_assert(U <= 12, "unroll table below covers twelve periods");
      period(IntTag<0>{});
      if constexpr (U > 1) period(IntTag<1>{});
      if constexpr (U > 2) period(IntTag<2>{});
      if constexpr (U > 3) period(IntTag<3>{});
      if constexpr (U > 4) period(IntTag<4>{});
      if constexpr (U > 5) period(IntTag<5>{});
      if constexpr (U > 6) period(IntTag<6>{});
      if constexpr (U > 7) period(IntTag<7>{});
      if constexpr (U > 8) period(IntTag<8>{});
      if constexpr (U > 9) period(IntTag<9>{});
      if constexpr (U > 10) period(IntTag<10>{});
      if constexpr (U > 11) period(IntTag<11>{});
    }
  }
  for (; t + STAGES < KT; ++t) {
    __builtin_amdgcn_s_waitcnt((PWAIT & 0xF) | (((PWAIT >> 4) & 0x3) << 14) | 0x0070);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    conv_period_begin();
    const uint32_t dst = stage_of(t);
    const uint32_t sa1 = stage_of(t + 1), sb1 = sa1 + C::A_BYTES;
    if constexpr (FAST) {
      end_slab(sa1, sb1, Yes{}, dst, Par0{}, Yes{});
      inner_steps(sa1, sb1, Yes{}, dst, Par0{});
      dma_advance();
    } else {
      // slab t + STAGES: fetched into registers now, written to the freed slot after this period's MFMAs; the
      // writes have to be in LDS before the next barrier lets anyone read them
      i32x4 ra[GEN_NA], rb[GEN_NB];
      gen_fetch(kt0 + t + STAGES, tid, ra, rb);
      end_slab(sa1, sb1, No{}, 0u, Par0{}, Yes{});
      inner_steps(sa1, sb1, No{}, 0u, Par0{});
      gen_store(dst, tid, ra, rb);
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    }
  }
  // (2) ring draining: nothing left to issue
  for (; t + 1 < KT; ++t) {
    __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    conv_fixup();      // CONV: the last slab that was issued has landed; nothing reads it before the next barrier
    const uint32_t sa1 = stage_of(t + 1), sb1 = sa1 + C::A_BYTES;
    end_slab(sa1, sb1, No{}, 0u, Par0{}, Yes{});
    inner_steps(sa1, sb1, No{}, 0u, Par0{});
  }
  // (3) last k step of the final slab
  if (KT > 0) {
    if constexpr (PAIR) {
      cross_step(0u, 0u, No{}, No{}, 0u);
    } else {
#pragma unroll
      for (int x = 0; x < NMMA; ++x) mma_one(LAST, x);
    }
  }
  };

  // Ping-pong form of the K loop (TNX_PINGPONG builds).  The waves 0..NW/2-1 ("lead") and NW/2..NW-1 share the SIMDs
  // pairwise.  Time runs in phases 0..2*KT, a workgroup barrier before each; slab v takes two of them:
  //   phase 2v     lead: reads both k steps' fragments of slab v from LDS      other: the MFMAs of slab v-1
  //                both: issue their DMA ops of slab v+1 into the slot slab v-1 has left (read last in phase 2v-1)
  //   phase 2v+1   lead: the MFMAs of slab v, priority raised                   other: reads slab v; all wait for the DMA
  // and phase 2*KT for the second group's last slab.  Each group runs its own straight loop; both execute 2*KT+1
  // barriers.  Needs an even KT >= 2 (the prologue has issued slabs 0 and 1); the caller falls back to k_loop().
  auto pingpong_loop = [&]() __attribute__((always_inline)) {
    constexpr int NRD = C::KSTEPS * NREAD, NMM = C::KSTEPS * NMMA;
    auto load_phase = [&](uint32_t sa, auto with_dma, uint32_t dst) __attribute__((always_inline)) {
      constexpr bool WITH_DMA = decltype(with_dma)::value;
      // opaque slot base: the lane addresses of the phase are formed here and die with it, instead of one set per
      // slot living in registers through every phase
      asm volatile("" : "+s"(sa));
      const uint32_t sb = sa + C::A_BYTES;
#pragma unroll
      for (int i = 0; i < NRD; ++i) {
        if (TNX_PINGPONG != 3) read_one(i / NREAD, i % NREAD, sa, sb, i / NREAD);
        if constexpr (WITH_DMA) {
#pragma unroll
          for (int q = i * C::LPW / NRD; q < (i + 1) * C::LPW / NRD; ++q) if (TNX_PINGPONG != 4) dma_op(q, dst);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (WITH_DMA) dma_advance();
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the slot may be refilled after the next barrier
    };
    auto mma_phase = [&](auto with_dma, uint32_t dst) __attribute__((always_inline)) {
      constexpr bool WITH_DMA = decltype(with_dma)::value;
      constexpr int HALF = NMM / 2;         // the refill goes out under the first half of the MFMAs
      if (TNX_PINGPONG != 2) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < NMM; ++i) {
        if (TNX_PINGPONG != 5) mma_one(i / NMMA, i % NMMA);
        if constexpr (WITH_DMA) {
          if (i < HALF) {
#pragma unroll
            for (int q = i * C::LPW / HALF; q < (i + 1) * C::LPW / HALF; ++q) if (TNX_PINGPONG != 4) dma_op(q, dst);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_s_setprio(0);
      if constexpr (WITH_DMA) dma_advance();
    };
    auto phase_barrier = [&]() __attribute__((always_inline)) {
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    const uint32_t s0 = lds0, s1 = lds0 + C::STAGE_BYTES;
    if (wave < NW / 2) {
      for (int v = 0; v < KT; v += 2) {
        phase_barrier();                                             // phase 2v
        if (v > 0) load_phase(s0, Yes{}, s1); else load_phase(s0, No{}, 0u);
        phase_barrier();                                             // 2v+1
        mma_phase(No{}, 0u);
        TNX_WAIT_VM(0);
        phase_barrier();                                             // 2v+2
        if (v + 2 < KT) load_phase(s1, Yes{}, s0); else load_phase(s1, No{}, 0u);
        phase_barrier();                                             // 2v+3
        mma_phase(No{}, 0u);
        TNX_WAIT_VM(0);
      }
      phase_barrier();                                               // phase 2*KT: the other group's last MFMAs
    } else {
      phase_barrier();                                               // phase 0: nothing to multiply yet
      for (int v = 0; v + 2 < KT; v += 2) {
        phase_barrier();                                             // 2v+1
        load_phase(s0, No{}, 0u);
        TNX_WAIT_VM(0);
        phase_barrier();                                             // 2v+2: slab v, and the DMA of slab v+2
        mma_phase(Yes{}, s0);
        phase_barrier();                                             // 2v+3
        load_phase(s1, No{}, 0u);
        TNX_WAIT_VM(0);
        phase_barrier();                                             // 2v+4: slab v+1, and the DMA of slab v+3
        mma_phase(Yes{}, s1);
      }
      phase_barrier();                                               // the last two slabs: nothing left to fetch
      load_phase(s0, No{}, 0u);
      TNX_WAIT_VM(0);
      phase_barrier();
      mma_phase(No{}, 0u);
      phase_barrier();
      load_phase(s1, No{}, 0u);
      phase_barrier();                                               // phase 2*KT
      mma_phase(No{}, 0u);
    }
  };
  typedef typename OutOf<T>::type O;
  if constexpr (!PERSIST) {
    if (KT > 0) {
      issue_prologue();
      if (KT >= STAGES) { TNX_WAIT_VM((STAGES - 1) * C::LPW); } else { TNX_WAIT_VM(0); }
    }
    if (PINGPONG_TILE && KT >= 2 && (KT & 1) == 0) pingpong_loop();
    else k_loop();
    if constexpr (FAST && !CONV && !GATHER && !PAIR) {
      if (tail_here) {
        // the left-out slab: every wave is done with the ring, slot 0 takes it, one slab of MFMAs follows
        __syncthreads();
        load_tail(kt1 - 1, stage_of(0), wave * 64 + lane);
        __syncthreads();
        const uint32_t sa = stage_of(0), sb = sa + C::A_BYTES;
#pragma unroll
        for (int ks = 0; ks < C::KSTEPS; ++ks) {
          if (ks > 0 && p.k - (int64_t)(kt1 - 1) * BK <= ks * (BK / C::KSTEPS)) break;      // zeros
#pragma unroll
          for (int idx = 0; idx < NREAD; ++idx) read_one(0, idx, sa, sb, ks);
#pragma unroll
          for (int x = 0; x < NMMA; ++x) mma_one(0, x);
        }
      }
    }

    // ---- epilogue ------------------------------------------------------------
    // every wave is done with the slabs before the LDS is reused for the output strips
    __syncthreads();
    const int64_t gm0 = m0 + wy * C::WTM;
    const int64_t gn0 = n0 + wx * C::WTN;
    const uint32_t strip = lds0 + wave * EpiStage<C>::WAVE_BYTES;
    // Float32 pairs: the lane again, from nothing that is older.  What the epilogue works out from it is else worked out before the K
    // loop, whose operands share a part of it, and carried through -- 256x256, k-contiguous B: 52 registers spilled, seven reloads per
    // two slabs, 3019 x 6592 x 5248 555 us; now none, 479.  Likewise the 256x256 tiles of four waves and one k step per slab (16-bit, four
    // slots: 4096^3 164 -> 141 us, three: 125 -> 120, two: even; int8 with two: 165 -> 118, with three and four 1 and 5 % the other way).
    // Tiles with registers to spare lose by it (4032 x 1696 x 1536 bf16 on 128x256 22.5 -> 23.7), and so does the one of four waves and
    // two k steps, which spills outside its loop only (8192^3 698 -> 717).
    constexpr bool NEW_LANE = PAIR || (C::KSTEPS == 1 && NW == 4 && BM == 256 && BN == 256 && (ES == 2 || STAGES == 2));
    const int elane = NEW_LANE ? __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) : lane;
    if constexpr (CONV) {
      if (p.out_dtype == DT_F32) epilogue_store_conv<T, C, OutF32>(acc, p.c, strip, elane, (int)gm0, (int)gn0, p.cv);
      else epilogue_store_conv<T, C, O>(acc, p.c, strip, elane, (int)gm0, (int)gn0, p.cv);
      return;
    }
    // `sums`: the wave's accumulators, or what the slices of a cut tile add up to.  The output type: the input's own
    // 16-bit type (int32 for int8), or binary32 where that epilogue is built.
    auto finish = [&](auto& sums) __attribute__((always_inline)) {
      auto as = [&](auto otag) __attribute__((always_inline)) {
        typedef typename decltype(otag)::type OT;
        if constexpr (GATHER)
          epilogue_store_conv<T, C, OT>(sums, p.c, strip, elane, (int)gm0, (int)gn0, p.cv);
        else if (p.epilogue == EPI_NONE)
          epilogue_store<T, C, OT, false, MULTI>(sums, p.c, strip, elane, gm0, gn0, p.m, p.n, p.scm, p.scn, p.c_row_ok, 0,
                                                 p.cv.bias, p.cv.bias_dtype);
        else
          epilogue_store<T, C, OT, true>(sums, p.c, strip, elane, gm0, gn0 >> 1, p.m, p.n >> 1, p.scm, p.scn, p.c_row_ok,
                                         p.epilogue);
      };
      if constexpr (PAIR) {
        as(TypeTag<OutF32>{});
      } else if constexpr (GATHER || f32_out_tile<T, C>()) {
        if (p.out_dtype == DT_F32) as(TypeTag<OutF32>{});
        else as(TypeTag<O>{});
      } else {
        as(TypeTag<O>{});
      }
    };
    if constexpr (!CONV) {
      if (cut) {
        // workspace after the counters: [slice][cut tile][wave][group][lane] 16-byte elements
        constexpr bool APART = RING_OR_STRIPS >= EpiStage<C>::BYTES + 16;
        const int ncut = ntiles - p.split_tile0, ctile = logical - p.split_tile0;
        const int64_t slice_stride = (int64_t)ncut * BM * BN * 4;
        uint8_t* wave0 = p.ws + WS_COUNTER_BYTES + ((int64_t)ctile * NW + wave) * (C::WTM * C::WTN * 4);
        const bool atomic = !GATHER && p.atomic_reduce != 0;
        if (!splitk_arrive<T, C, APART>(acc, wave0 + (atomic ? 0 : split * slice_stride), elane, gm0, p.m, (int*)p.ws + ctile,
                                        (int*)(smem + (APART ? EpiStage<C>::BYTES : 0)), p.split_k, atomic))
          return;
        acc_t sums[TM][TN];          // (not `acc`: two definitions that meet again spill in the tiles that use every register)
        collect_slices<C>(sums, SliceSrc{wave0, (uint32_t)slice_stride, atomic ? 1 : p.split_k, atomic}, elane, p.m - gm0);
        finish(sums);
        return;
      }
    }
    finish(acc);
  } else {
    // ---- persistent: this workgroup walks tiles blockIdx.x, blockIdx.x + gridDim.x, ... ------------
    // The host launches it only with KT >= STAGES.  While the epilogue of a tile runs, the first
    // STAGES slabs of the next tile are already on their way into the ring, and the epilogue's
    // stores drain under the next tile's first K slabs.  vmcnt retires in issue order, so
    // "at most X operations outstanding" means the X youngest: after an epilogue these are its
    // stores, and everything older -- the next tile's prologue -- has landed.  X may therefore
    // include the stores only when their number is known exactly (a tile fully inside C with
    // 16-byte stores); otherwise it is the (STAGES - 1) slabs of the prologue that may stay in
    // flight, as for the first tile.
    const uint32_t strip = lds0 + C::LDS_BYTES + wave * PairStrip<C>::WAVE_BYTES;
    constexpr int X_FIRST = (STAGES - 1) * C::LPW;
    constexpr int NST_PLAIN = PairEpilogue<T, C, O, false>::STORES, NST_GLU = PairEpilogue<T, C, O, true>::STORES;
    constexpr int X_PLAIN = X_FIRST + NST_PLAIN > 63 ? 63 : X_FIRST + NST_PLAIN;
    constexpr int X_GLU = X_FIRST + NST_GLU > 63 ? 63 : X_FIRST + NST_GLU;
    const bool glu = p.epilogue != EPI_NONE;
    issue_prologue();
    TNX_WAIT_VM(X_FIRST);
    for (int id = blockIdx.x; id < ntiles; id += gridDim.x) {
      k_loop();
      // every wave is done with the ring: it can take the next tile's first slabs
      __syncthreads();
      const int64_t gm0 = m0 + wy * C::WTM;
      const int64_t gn0 = n0 + wx * C::WTN;
      const bool full = p.c_vec_ok && m0 + BM <= p.m && n0 + BN <= p.n;
      const int next = id + gridDim.x;
      if (next < ntiles) {
        int nm, nn;
        locate(next, &nm, &nn);
        place_tile(nm, nn);
        issue_prologue();
      }
      // The epilogue's per-lane offsets depend only on the lane: left alone, the compiler computes them once
      // before the tile loop and keeps them in registers across every K loop, which spills.  An opaque copy of
      // the lane index ties them to this iteration.
      int lane_e = lane;
      asm volatile("" : "+v"(lane_e));
      if (!glu) {
        if (full) epilogue_store_pairs<T, C, O, false, true>(acc, p.c, strip, lane_e, gm0, gn0, p.m, p.n, p.scm, p.scn, true, 0);
        else epilogue_store_pairs<T, C, O, false, false>(acc, p.c, strip, lane_e, gm0, gn0, p.m, p.n, p.scm, p.scn, p.c_vec_ok, 0);
      } else {
        if (full) epilogue_store_pairs<T, C, O, true, true>(acc, p.c, strip, lane_e, gm0, gn0 >> 1, p.m, p.n >> 1, p.scm, p.scn, true, p.epilogue);
        else epilogue_store_pairs<T, C, O, true, false>(acc, p.c, strip, lane_e, gm0, gn0 >> 1, p.m, p.n >> 1, p.scm, p.scn, p.c_vec_ok, p.epilogue);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{};
      if (next < ntiles) {
        if (!full) { TNX_WAIT_VM(X_FIRST); }
        else if (glu) { TNX_WAIT_VM(X_GLU); }
        else { TNX_WAIT_VM(X_PLAIN); }
      }
    }
  }
}

}  // namespace tnx
