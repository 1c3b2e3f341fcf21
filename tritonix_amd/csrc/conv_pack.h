// Operands of a conv2d forward laid out for the k-contiguous GEMM kernel (gemm_tile_kernel<..., GATHER>).
//
//   input  [batch][c_in][h][w]        ->  [batch][rows][cols][terms * cp]   zero padding written out
//   weight [c_out][c_in][fh][fw]      ->  [c_out][fh * fw][terms * cp], rows zero-filled to whole K slabs
//
// with cp = c_in rounded up to 8.  16-bit operands have one term; float32 operands are cut into bf16 terms for
// hi hi + hi lo + lo hi: as a head and a tail in blocks of 32 channels (two terms; the PAIR form of the GEMM kernel, a
// non-finite element having +-1 for its head and itself for its tail), or, where padding the channels to 32 costs more
// than the third copy, as three terms -- input [hi | hi' | lo], weight [hi | lo | hi'], hi' being hi without its
// infinities and NaNs (the split of tnx_split_f32).
//
// What it buys: the im2col loaders gather the same input element once per filter tap with address arithmetic and edge
// masks in the MFMA stream; after this pass a tap is a constant added to an address.  One launch does both operands.
// Bound by memory traffic: each input element is read once and written once (plus the borders).  A thread moves 8
// channels x 8 columns: eight 16-byte loads along the rows, an 8x8 transpose of 16-bit elements in registers (32 byte
// permutes, no LDS), eight 16-byte stores along the channels; 8 lanes are 8 neighbouring channel groups, the 8 groups of
// lanes 8 neighbouring column chunks, so loads and stores both move 128-byte runs.  256 channels of 56x56, batch 32, bf16:
// 17.9 us for 51 MB in and 55 MB out, 5.9 TB/s (a plain copy of that size: 15.7 us); with the blocks dealt round-robin to
// the XCDs 25.3 us, with non-temporal loads 31 us.
#pragma once
#include "gemm_tile.h"

namespace tnx {

struct PackParams {
  const uint8_t* x;
  const uint8_t* w;
  uint8_t* xp;
  uint8_t* wp;
  int* counters;               // arrival counters of a K cut, cleared here (null: none)
  int ncounters;
  int c_in, h_in, w_in, taps;
  int rows, cols;              // of the packed image
  int step_h, step_w;          // input rows / columns from one packed row / column to the next
  int pad_h, pad_w;
  int cp8, chunks, chunks_pad; // channel groups of 8 per term; k chunks of a weight row, and up to whole slabs
  int wchunks;                 // column chunks of 8 per packed row, counted from column `lead` (the padding before it is
  int lead;                    // written with the first chunk, that after the last input column with the last)
  bool whole;                  // a tap's channels are whole K slabs
  int cgb;                     // blocks of 8 channel groups
  int x_items, w_items;        // input: (image, row, column chunk) triples; weight: (c_out, chunk) pairs
  int x_elems;                 // elements of the input
  unsigned w_blocks;           // workgroups [0, w_blocks) lay out the weight, the others the input
  FastDiv div_cgb, div_row, div_wchunks, div_cpt, div_cp8, div_chunks, div_taps;
};

// one element as its bf16 (or 16-bit) terms; side 0: input order, side 1: weight order
template <int SIDE> __device__ __forceinline__ void pack_terms(uint16_t v, uint16_t (&t)[1]) { t[0] = v; }
template <int SIDE> __device__ __forceinline__ void pack_terms(float v, uint16_t (&t)[3]) {
  const __bf16 hi = (__bf16)v;
  const float rest = v - (float)hi;
  const bool fin = __builtin_isfinite(rest) && __builtin_isfinite((float)hi);
  const uint16_t h = __builtin_bit_cast(uint16_t, hi), l = __builtin_bit_cast(uint16_t, (__bf16)rest);
  t[0] = h;
  t[SIDE == 0 ? 1 : 2] = fin ? h : (uint16_t)0;
  t[SIDE == 0 ? 2 : 1] = fin ? l : (uint16_t)0;
}
template <int SIDE> __device__ __forceinline__ void pack_terms(float v, uint16_t (&t)[2]) {
  const __bf16 hi = (__bf16)v;
  const float rest = v - (float)hi;
  const bool fin = __builtin_isfinite(rest) && __builtin_isfinite((float)hi);
  const __bf16 one = __builtin_signbit(v) ? (__bf16)-1.0f : (__bf16)1.0f;
  t[0] = __builtin_bit_cast(uint16_t, fin ? hi : one);
  t[1] = __builtin_bit_cast(uint16_t, fin ? (__bf16)rest : hi);
}
// chunk of term z of channel group cg among a pixel's (or filter tap's) chunks
template <int NT> __device__ __forceinline__ int term_chunk(int z, int cg, int cp8) {
  return NT == 2 ? (cg >> 2) * 8 + z * 4 + (cg & 3) : z * cp8 + cg;
}

template <class E, int NT>
__global__ __launch_bounds__(256) void conv_pack_kernel(PackParams p) {
  const int tid = threadIdx.x;
  if (blockIdx.x < p.w_blocks) {
    const int item = blockIdx.x * 256 + tid;
    if (p.counters && item < p.ncounters) p.counters[item] = 0;
    if (item >= p.w_items) return;
    const int co = (int)fd_div((uint32_t)item, p.div_chunks), k8 = item - co * p.chunks_pad;
    i32x4 v = {0, 0, 0, 0};
    if (k8 < p.chunks) {
      // k order: the channels of a filter tap together; or, where they are whole K slabs, the taps of 64 channels together
      // (the same input lines are then read again while they are still in the L2)
      int tap, r;
      if (p.whole) {
        const int slab = k8 >> 3, cs = (int)fd_div((uint32_t)slab, p.div_taps);
        tap = slab - cs * p.taps;
        r = cs * 8 + (k8 & 7);
      } else {
        tap = (int)fd_div((uint32_t)k8, p.div_cpt);
        r = k8 - tap * (p.cp8 * NT);
      }
      const int term = NT == 1 ? 0 : NT == 2 ? (r >> 2) & 1 : (int)fd_div((uint32_t)r, p.div_cp8);
      const int cg = NT == 2 ? (r >> 3) * 4 + (r & 3) : r - term * p.cp8;
      const E* src = (const E*)p.w + ((int64_t)co * p.c_in + cg * 8) * p.taps + tap;
      uint16_t o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint16_t t[NT];
        pack_terms<1>(cg * 8 + e < p.c_in ? src[(int64_t)e * p.taps] : (E)0, t);
        o[e] = t[0];
        if constexpr (NT == 2) o[e] = term == 0 ? t[0] : t[1];
        if constexpr (NT == 3) o[e] = term == 0 ? t[0] : term == 1 ? t[1] : t[2];
      }
      __builtin_memcpy(&v, o, 16);
    }
    *(i32x4*)(p.wp + (int64_t)item * 16) = v;
    return;
  }
  // neighbouring blocks on one XCD: a 128-byte run of a plane starts anywhere, so the cache lines at its ends are the
  // neighbour's too, and a second L2 would have to fetch them again
  const int wave = xcd_remap(blockIdx.x - p.w_blocks, gridDim.x - p.w_blocks, 8) * 4 + (tid >> 6), lane = tid & 63;
  const int jb = (int)fd_div((uint32_t)wave, p.div_cgb), cgblk = wave - jb * p.cgb;
  const int j = jb * 8 + (lane >> 3), cg = cgblk * 8 + (lane & 7);
  if (j >= p.x_items || cg >= p.cp8) return;
  const int row_all = (int)fd_div((uint32_t)j, p.div_wchunks), wc = j - row_all * p.wchunks;
  const int img = (int)fd_div((uint32_t)row_all, p.div_row), row = row_all - img * p.rows;
  const int h = row * p.step_h - p.pad_h, col0 = wc * 8 + p.lead, w0 = col0 * p.step_w - p.pad_w;
  E in[8][8];                                       // [channel][column]
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) in[c][e] = (E)0;
  if ((uint32_t)h < (uint32_t)p.h_in && w0 < p.w_in && w0 + 7 * p.step_w >= 0) {
    const int plane = p.h_in * p.w_in;
    const int o0 = ((img * p.c_in + cg * 8) * p.h_in + h) * p.w_in + w0;    // element of (channel 0, column 0)
    const E* src = (const E*)p.x;
    const int nch = p.c_in - cg * 8 < 8 ? p.c_in - cg * 8 : 8;
    const int lo = w0 < 0 ? -w0 : 0, hi = p.w_in - w0;                      // elements [lo, hi) of a unit-stride run lie in the row
    if (p.step_w == 1 && o0 >= 0 && o0 + (nch - 1) * plane <= p.x_elems - 8) {
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (c < nch) {
          struct __attribute__((packed, aligned(sizeof(E)))) Row { E v[8]; };
          const Row v = *(const Row*)(src + o0 + c * plane);
#pragma unroll
          for (int e = 0; e < 8; ++e) in[c][e] = v.v[e];
        }
      if (lo > 0 || hi < 8) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e < lo || e >= hi) {
#pragma unroll
            for (int c = 0; c < 8; ++c) in[c][e] = (E)0;
          }
      }
    } else if (p.step_w == 2 && w0 >= 0 && w0 + 16 <= p.w_in) {
#pragma unroll
      for (int c = 0; c < 8; ++c)
        if (c < nch) {
          struct __attribute__((packed, aligned(sizeof(E)))) Row { E v[16]; };
          const Row v = *(const Row*)(src + o0 + c * plane);
#pragma unroll
          for (int e = 0; e < 8; ++e) in[c][e] = v.v[2 * e];
        }
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (c < nch && (uint32_t)(w0 + e * p.step_w) < (uint32_t)p.w_in) in[c][e] = src[o0 + c * plane + e * p.step_w];
    }
  }
  uint8_t* dst = p.xp + ((int64_t)row_all * p.cols + col0) * (p.cp8 * NT) * 16;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (col0 + e >= p.cols) break;
    uint16_t o[NT][8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      uint16_t t[NT];
      pack_terms<0>(in[c][e], t);
#pragma unroll
      for (int z = 0; z < NT; ++z) o[z][c] = t[z];
    }
#pragma unroll
    for (int z = 0; z < NT; ++z) {
      i32x4 v;
      __builtin_memcpy(&v, o[z], 16);
      *(i32x4*)(dst + ((int64_t)e * (p.cp8 * NT) + term_chunk<NT>(z, cg, p.cp8)) * 16) = v;
    }
  }
  if (wc == 0)
    for (int col = -p.lead; col < 0; ++col)
#pragma unroll
      for (int z = 0; z < NT; ++z) *(i32x4*)(dst + ((int64_t)col * (p.cp8 * NT) + term_chunk<NT>(z, cg, p.cp8)) * 16) = i32x4{0, 0, 0, 0};
  if (wc == p.wchunks - 1)
    for (int col = 8; col0 + col < p.cols; ++col)
#pragma unroll
      for (int z = 0; z < NT; ++z) *(i32x4*)(dst + ((int64_t)col * (p.cp8 * NT) + term_chunk<NT>(z, cg, p.cp8)) * 16) = i32x4{0, 0, 0, 0};
}

}  // namespace tnx
