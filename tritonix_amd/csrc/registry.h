// Table of compiled tile kernels.  Each generated instance file contributes
// one array of KernelEntry; capi.hip looks a tile config up in the union.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_tile.h"

struct tnx_gemm_args;

namespace tnx {

typedef hipError_t (*launch_fn)(const GemmParams& p, unsigned grid, hipStream_t stream);

struct KernelEntry {
  int dtype, bm, bn, bk, nw, stages;
  int lds_bytes;
  launch_fn fast;     // DMA loader: row-major, 16-byte aligned, k % bk == 0
  launch_fn generic;  // element-wise loader: any strides / ragged k; may be null
  launch_fn persist;  // DMA loader, one workgroup per CU walking its tiles; may be null
  launch_fn fast_bt;  // DMA loader for k-contiguous B (stride_bk == 1, the `x @ w.t()` layout); may be null
  launch_fn conv;     // conv2d forward on the DMA loader (GemmParams::cv); may be null
  launch_fn fast_at;  // DMA loader for m-contiguous A (stride_am == 1, the `x.t() @ dy` layout), row-major B; may be null
  launch_fn pair[3];  // float32 products on head and tail slabs (gemm_tile_kernel<..., PAIR>): row-major B, k-contiguous B, m-contiguous A; may be null
};

// records the hipError_t behind a TNX_E_HIP for tnx_last_hip_error() (per thread)
void note_hip_error(int err);
// tnx_gemm with `batch` problems in one grid -- same A, problem i reads b + i * b_batch_bytes and writes
// c + i * c_batch_bytes -- and an optional bias per row of C, added to the fp32 sum before the rounding (float types).
// Uncut, non-persistent launches of tiles up to 128x128 only (multi_problem_tile).  conv2d's 1x1 layers are this GEMM,
// one problem per image.
struct GemmBatch {
  int batch;
  int64_t b_batch_bytes, c_batch_bytes;
  const void* bias;
  int bias_dtype;
};
// What the operands of a launch are.  PADDED: the rows of B (and of an m-contiguous A) are followed by readable memory up
// to a whole 16-byte chunk, so an N (M) that ends inside a chunk still takes the aligned loader.  PAIR: padded, and k
// holds the heads and tails of a float32 product in blocks of 32 (KernelEntry::pair).
// F32: float32 operands as they are, on the binary32 matrix instruction.
enum GemmForm { GEMM_PLAIN = 0, GEMM_PADDED = 1, GEMM_PAIR = 2, GEMM_F32 = 3 };
int gemm_launch(const tnx_gemm_args* a, const GemmBatch* extra, GemmForm form = GEMM_PLAIN);
// the status gemm_launch would return for these arguments, the workspace included, without launching
int gemm_check(const tnx_gemm_args* a, GemmForm form);
// whether the tile of `a` and the layout of its float32 operands have a kernel that multiplies them as they are
bool gemm_f32_direct(const tnx_gemm_args* a, bool any_base);
// whether the tile of `a` takes head and tail slabs, and whether it has the k-contiguous-B and m-contiguous-A loaders
void gemm_tile_layouts(const tnx_gemm_args* a, bool* pair, bool* bt, bool* at);
// waves and stages of a built tile with these dimensions that gemm_launch takes with a GemmBatch (eight waves and
// two ring slots first); false: none built
bool gemm_tile_for(int dtype, int bm, int bn, int bk, int* num_warps, int* num_stages);

// conv2d over a packed input (gemm_tile_kernel<..., GATHER>), block_k = 64: tiles of channels x pixels
struct GatherEntry {
  int dtype, bm, bn, nw, stages;
  launch_fn launch;
  launch_fn pair;     // float32 operands as head and tail slabs; bf16 entries only
};
struct GatherGroup {
  GatherEntry* entries;
  int count;
};

struct KernelGroup {
  KernelEntry* entries;
  int count;
};

template <class T, class C, bool FAST, bool PERSIST = false, bool BT = false, bool CONV = false, bool GATHER = false,
          bool AT = false, bool PAIR = false>
hipError_t launch_tile(const GemmParams& p, unsigned grid, hipStream_t stream) {
  static_assert(GATHER ? C::VALID_GATHER : C::VALID, "tile configuration is not buildable");
  constexpr bool PLAIN = FAST && !CONV && !GATHER;
  typename KernelParams<PLAIN>::type q;
  if constexpr (PLAIN) {
    if (!plain_params(p, BT, AT, C::ES, &q)) return hipErrorInvalidValue;
  } else {
    q = p;
    set_order_divisors(&q);
  }
  return launch_kernel((const void*)&gemm_tile_kernel<T, C, FAST, PERSIST, BT, CONV, GATHER, AT, PAIR>, grid, C::THREADS, 0, stream, &q);
}

// The persistent variant exists for the four-wave tiles from 128x128 to 256x128 / 128x256: their ring leaves
// room for the epilogue's own strips (MI rows of 256 bytes per wave) inside the 160 KiB of one CU, and a wave's
// accumulators take at most 128 registers, so the state the tile loop carries still fits the register file
// (with the 256 accumulator registers of a 256x256 tile it does not: the compiler spills inside the K loop).
template <class C> constexpr bool persist_ok() {
  return C::NW == 4 && C::BM >= 128 && C::BN >= 128 && C::TN % PairStrip<C>::TPP == 0 &&
         C::TM * C::TN * C::ACC_N <= 128 && C::LDS_BYTES + PairStrip<C>::BYTES <= 163840;
}
template <class T, class C, bool OK = persist_ok<C>()> struct PersistLaunch {
  static constexpr launch_fn fn = nullptr;
};
template <class T, class C> struct PersistLaunch<T, C, true> {
  static constexpr launch_fn fn = &launch_tile<T, C, true, true>;
};

// skinny kernel (gemm_skinny.h): tile 16 x 32 x 32, eight waves, split_k == 8 inside the workgroup,
// num_stages = ring depth per wave.  Null when that depth / dtype is not built.
launch_fn skinny_lookup(int dtype, int ring);
constexpr int SKINNY_BM = 16, SKINNY_BN = 32, SKINNY_BK = 32, SKINNY_NW = 8, SKINNY_SPLIT = 8;
constexpr int SKINNY_STEP_BYTES = 3072;

// The k-contiguous-B variant exists for the tiles whose K slab is one 128-byte line per row (the tiles the
// built-in choice uses).
template <class C> constexpr bool bt_ok() { return C::BK * C::ES == 128; }
template <class T, class C, bool OK = bt_ok<C>()> struct BtLaunch {
  static constexpr launch_fn fn = nullptr;
};
template <class T, class C> struct BtLaunch<T, C, true> {
  static constexpr launch_fn fn = &launch_tile<T, C, true, false, true>;
};

// The conv2d variant exists for the three-slot, eight-wave 16-bit tiles 128x128, 256x128 and 128x256 with a 128-byte K
// slab (with four waves it was measured 15-20 % slower, and 256x256 then has no registers left for the loader's state;
// three slots of 256x256 do not fit the LDS; a 64-channel tile was measured and loses to the
// register-staged kernel).  The second half of a period must have room for the slotted fix-up of all B ops.
template <class C> constexpr bool conv_ok() {
  return C::ES == 2 && C::NW == 8 && C::KSTEPS * C::TM * C::TN >= 16 &&
         C::KSTEPS * C::TM * C::TN / 2 > C::B_LPW + (C::KSTEPS * C::TM * C::TN >= 32 ? 6 : 3) + 1 && C::STAGES == 3 && C::BK == 64 &&
         C::BM >= 128 && C::BN >= 128 && C::TM * C::TN * C::ACC_N <= 128 && (C::NW * 64) % C::CPR_B == 0;
}
template <class T, class C, bool OK = conv_ok<C>()> struct ConvLaunch {
  static constexpr launch_fn fn = nullptr;
};
template <class T, class C> struct ConvLaunch<T, C, true> {
  static constexpr launch_fn fn = &launch_tile<T, C, true, false, false, true>;
};

// The m-contiguous-A variant exists for the tiles the built-in choice proposes, with the waves and slots it gives them.
// (64 rows of int8 are too short for the transposing read; the 256x256 tile takes eight waves for every K: with four it
// spills.)
template <class C> constexpr bool at_ok() {
  return C::BK * C::ES == 128 && C::VALID_AT &&
         (C::ES == 4 || (C::BM == 256 && C::BN == 256 && C::NW == 8 && C::STAGES == 2) || (C::BM == 256 && C::BN == 128 && C::NW == 4 && C::STAGES == 3) ||
          (C::BM == 128 && C::BN == 128 && C::NW == 8 && C::STAGES == 3) || (C::BM == 64 && C::BN == 128 && C::NW == 8 && C::STAGES == 3) ||
          (C::BM == 64 && C::BN == 64 && C::NW == 4 && C::STAGES == 4) || (C::BM == 192 && C::BN == 192 && C::NW == 8 && C::STAGES == 3) ||
          ((C::BM == 192 || C::BN == 192) && C::BM != C::BN && C::NW == 8 && C::STAGES == 2));
}
template <class T, class C, bool PAIR = false, bool OK = at_ok<C>()> struct AtLaunch {
  static constexpr launch_fn fn = nullptr;
};
template <class T, class C, bool PAIR> struct AtLaunch<T, C, PAIR, true> {
  static constexpr launch_fn fn = &launch_tile<T, C, true, false, false, false, false, true, PAIR>;
};

// The float32 variant exists for the tiles the built-in choice proposes for float32 problems.
template <class T, class C> constexpr bool pair_ok() {
  return T::ID == DT_BF16 && C::BK == 64 &&
         ((C::NW == 8 && (C::BM == 256 || C::BM == 192) && (C::BN == 256 || C::BN == 192) && C::STAGES == (C::BM == 192 && C::BN == 192 ? 3 : 2)) ||
          (C::BM == 128 && C::BN == 128 && C::STAGES == 3) || (C::NW == 8 && C::BM == 64 && C::BN == 128 && C::STAGES == 3) ||
          (C::NW == 4 && C::BM == 64 && C::BN == 64 && C::STAGES == 4));
}
template <class T, class C, bool OK = pair_ok<T, C>()> struct PairLaunch {
  static constexpr launch_fn nn = nullptr, bt = nullptr, at = nullptr;
};
template <class T, class C> struct PairLaunch<T, C, true> {
  static constexpr launch_fn nn = &launch_tile<T, C, true, false, false, false, false, false, true>;
  static constexpr launch_fn bt = &launch_tile<T, C, true, false, true, false, false, false, true>;
  static constexpr launch_fn at = AtLaunch<T, C, true>::fn;
};

// The element-wise loader is built only for the tiles that ask for it (a conditional expression would instantiate
// the kernel for every tile and merely not point at it).
template <class T, class C, bool WANTED> struct GenericLaunch {
  static constexpr launch_fn fn = nullptr;
};
template <class T, class C> struct GenericLaunch<T, C, true> {
  static constexpr launch_fn fn = &launch_tile<T, C, false>;
};

template <class T, class C, bool OK = T::ID == DT_BF16> struct GatherPairLaunch {
  static constexpr launch_fn fn = nullptr;
};
template <class T, class C> struct GatherPairLaunch<T, C, true> {
  static constexpr launch_fn fn = &launch_tile<T, C, true, false, true, false, true, false, true>;
};

#define TNX_GATHER_ENTRY(TAG, BM, BN, NW, ST)                                                                      \
  {TAG::ID, BM, BN, NW, ST, &launch_tile<TAG, TileCfg<TAG, BM, BN, 64, NW, ST>, true, false, true, false, true>,  \
   GatherPairLaunch<TAG, TileCfg<TAG, BM, BN, 64, NW, ST>>::fn}

#define TNX_ENTRY(TAG, BM, BN, BK, NW, ST, GENERIC)                                                          \
  {TAG::ID, BM, BN, BK, NW, ST, TileCfg<TAG, BM, BN, BK, NW, ST>::LDS_BYTES,                                 \
   &launch_tile<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>, true>,                                                \
   GenericLaunch<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>, GENERIC>::fn,                                        \
   PersistLaunch<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>>::fn, BtLaunch<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>>::fn,     \
   ConvLaunch<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>>::fn, AtLaunch<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>>::fn,         \
   {PairLaunch<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>>::nn, PairLaunch<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>>::bt,           \
    PairLaunch<TAG, TileCfg<TAG, BM, BN, BK, NW, ST>>::at}}

}  // namespace tnx
