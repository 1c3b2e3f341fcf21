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
// lanes 8 neighbouring column chunks (but see pack_cg_bits), so loads and stores both move 128-byte runs.  256 channels of 56x56, batch 32, bf16:
// 17.9 us for 51 MB in and 55 MB out, 5.9 TB/s (a plain copy of that size: 15.7 us); with the blocks dealt round-robin to
// the XCDs 25.3 us, with non-temporal loads 31 us.
//
// Small inputs are bound by the latency of one wave instead, so its loads do not wait for one another and its lanes share one
// path (see fetch): with a condition around each load, layers took, both launches in a graph, 59 -> 64 channels of 14x14, 3x3,
// batch 4 10.6 us, now 8.5; 512 -> 512 of 7x7, one image 15.4, 13.0; with a stride of two, where half of the lanes went element by
// element, 384 -> 256 of 28x28, 1x1, batch 8 13.8, 9.7, and 896 -> 2048, batch 128 192, 164.
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
  int cgb;                     // blocks of as many channel groups as a wave has side by side (pack_cg_bits)
  int x_items, w_items;        // input: (image, row, column chunk) triples; weight: (c_out, chunk) pairs
  int x_elems;                 // elements of the input
  unsigned w_blocks;           // workgroups [0, w_blocks) lay out the weight, the others the input
  FastDiv div_cgb, div_row, div_wchunks, div_cpt, div_cp8, div_chunks, div_taps;
};

// Lanes of a wave: neighbouring channel groups by neighbouring column chunks, 8 x 8 or, with a single channel group, 1 x 64.  (With 8 x 8
// there too seven lanes of eight had nothing to do, in eight times the waves, each of which fetches the kernel's 20 KB of
// instructions: float32, both launches, 3 -> 80 channels of 28x28, 1x1, one image 13.4 -> 8.3 us; 5 -> 16 of 56x56, 3x3, batch 128 44.0 -> 36.3.)
__host__ __device__ constexpr int pack_cg_bits(int cp8) { return cp8 == 1 ? 0 : 3; }

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

// Eight elements from `at` on, or from the nearest place where all eight lie inside [0, elems), elems >= 8 ...
template <class E> constexpr int RUN = 2 * sizeof(E);                     // 32-bit words of eight elements
template <class E> __device__ __forceinline__ void load_run(uint32_t* v, const E* src, int at, int elems) {
  struct __attribute__((packed, aligned(sizeof(E)))) Run { uint32_t v[RUN<E>]; };
  const Run r = *(const Run*)(src + (at < 0 ? 0 : at > elems - 8 ? elems - 8 : at));
#pragma unroll
  for (int i = 0; i < RUN<E>; ++i) v[i] = r.v[i];
}
// ... and those of them that do exist back at their index.
template <class E> __device__ __forceinline__ void turn_run(uint32_t* v, int at, int elems) {
  constexpr int W = RUN<E>;
  const int d = at - (at < 0 ? 0 : at > elems - 8 ? elems - 8 : at);
  if (d == 0 || d <= -8 || d >= 8) return;                                // (wholly outside: nothing to put back)
#pragma unroll
  for (int by = 1; by < 8; by *= 2) {
    uint32_t t[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
      if (W == 8) t[i] = v[(i + by) & 7];
      else t[i] = by == 1 ? v[i] >> 16 | v[(i + 1) & 3] << 16 : v[(i + by / 2) & 3];
    }
#pragma unroll
    for (int i = 0; i < W; ++i) v[i] = d & by ? t[i] : v[i];
  }
}

// UNIT: step_w is 1 (77 registers instead of 116, float32 128 instead of 162: one kernel for both lost 1 to 5 % in float32)
template <class E, int NT, bool UNIT>
__global__ __launch_bounds__(256, UNIT ? 1 : 3) void conv_pack_kernel(PackParams p) {
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
      const E* src = (const E*)p.w + (int64_t)co * p.c_in * p.taps + tap;
      E v8[8] = {};                                   // all loads before the first wait: a channel that does not exist repeats the last one
      if (cg * 8 < p.c_in) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v8[e] = src[(int64_t)(cg * 8 + e < p.c_in ? cg * 8 + e : p.c_in - 1) * p.taps];
      }
      uint16_t o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint16_t t[NT];
        pack_terms<1>(cg * 8 + e < p.c_in ? v8[e] : (E)0, t);
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
  const int cg_bits = pack_cg_bits(p.cp8), j = (jb << (6 - cg_bits)) + (lane >> cg_bits), cg = (cgblk << cg_bits) + (lane & ((1 << cg_bits) - 1));
  if (j >= p.x_items || cg >= p.cp8) return;
  const int row_all = (int)fd_div((uint32_t)j, p.div_wchunks), wc = j - row_all * p.wchunks;
  const int img = (int)fd_div((uint32_t)row_all, p.div_row), row = row_all - img * p.rows;
  const int step_w = UNIT ? 1 : p.step_w, h = row * p.step_h - p.pad_h, col0 = wc * 8 + p.lead, w0 = col0 * step_w - p.pad_w;
  constexpr int W = RUN<E>;
  uint32_t raw[8][W];                               // [channel][column], two 16-bit columns a word
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int i = 0; i < W; ++i) raw[c][i] = 0;
  if ((uint32_t)h < (uint32_t)p.h_in && w0 < p.w_in && w0 + 7 * step_w >= 0 && cg * 8 < p.c_in) {
    const int plane = p.h_in * p.w_in;
    const int o0 = ((img * p.c_in + cg * 8) * p.h_in + h) * p.w_in + w0;    // element of (channel 0, column 0)
    const E* src = (const E*)p.x;
    const int nch = p.c_in - cg * 8 < 8 ? p.c_in - cg * 8 : 8;
    auto in_row = [&](int e) { return (uint32_t)(w0 + e * step_w) < (uint32_t)p.w_in; };
    // what was read in the place of columns outside the row and of channels that do not exist
    auto clear = [&](auto nc) {
      constexpr int NC = nc;
      if (w0 < 0 || w0 + 7 * step_w >= p.w_in) {
#pragma unroll
        for (int i = 0; i < W; ++i) {
          const uint32_t keep = W == 8 ? (in_row(i) ? ~0u : 0u) : (in_row(2 * i) ? 0xffffu : 0u) | (in_row(2 * i + 1) ? 0xffff0000u : 0u);
#pragma unroll
          for (int c = 0; c < NC; ++c) raw[c][i] &= keep;
        }
      }
      if (nch < NC) {
#pragma unroll
        for (int c = 1; c < NC; ++c)
#pragma unroll
          for (int i = 0; i < W; ++i) raw[c][i] = c < nch ? raw[c][i] : 0u;
      }
    };
    constexpr std::integral_constant<int, 8> eight;
    if ((UNIT || step_w == 2) && p.x_elems >= 8) {
      // All loads are on their way before the first is waited for, and no lane takes another path at the edges: a load under a
      // condition of its own is waited for at the condition's end, eight latencies in a row.  So for channels that do not exist
      // and runs past the row all lanes read the input's first elements, a run that would leave the input is moved inside it and
      // turned back, and what lies outside the row is cleared.
      auto at = [&](int c) { return c < nch ? o0 + c * plane : 0; };
      const bool edge = o0 < 0 || o0 + (nch - 1) * plane + 8 * (step_w - 1) > p.x_elems - 8;
      // NC channels, every STEP-th element of RUNS runs
      auto fetch = [&](auto nc, auto step, auto runs) {
        constexpr int NC = nc, STEP = step, RUNS = runs, CB = RUNS == 2 && W == 8 ? 2 : NC;   // channels at a time, as the registers allow
        auto at_run = [&](int c, int r) { return r == 0 || w0 + 8 < p.w_in ? at(c) + 8 * r : 0; };
#pragma unroll
        for (int c0 = 0; c0 < NC; c0 += CB) {
          uint32_t t[CB][RUNS * W];
#pragma unroll
          for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int r = 0; r < RUNS; ++r) load_run<E>(t[c] + r * W, src, at_run(c0 + c, r), p.x_elems);
          if (edge) {
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
              for (int r = 0; r < RUNS; ++r) turn_run<E>(t[c] + r * W, at_run(c0 + c, r), p.x_elems);
          }
#pragma unroll
          for (int c = 0; c < CB; ++c)
#pragma unroll
            for (int i = 0; i < W * RUNS / STEP; ++i)
              raw[c0 + c][i] = STEP == 1 ? t[c][i] : W == 8 ? t[c][2 * i] : (t[c][2 * i] & 0xffffu) | t[c][2 * i + 1] << 16;
        }
        clear(nc);
      };
      // (rows that one run covers need no second, inputs of few channels no repeats)
      constexpr std::integral_constant<int, 1> one;
      constexpr std::integral_constant<int, 2> two;
      constexpr std::integral_constant<int, 4> four;
      if constexpr (UNIT) {
        if (p.c_in <= 4) fetch(four, one, one);
        else fetch(eight, one, one);
      } else {
        if (p.w_in + p.pad_w <= 8) fetch(eight, two, one);
        else fetch(eight, two, two);
      }
    } else {
      // Wider steps, and inputs shorter than a run: element by element, columns that a lane has not in its row read at the row's ends,
      // channels that do not exist in the first one's place.  Up to two waves of this pass on every CU (float32: one) a wave's latency
      // counts: all loads on their way before the first is waited for, but those of columns that no lane has.  With more it is the
      // lines that the L1 keeps until their next column is read: a channel at a time, or in float32, whose words need no packing, all
      // channels at once without a condition.  1x1 layers at steps of 3 and 4, both launches: 300 -> 256 channels of 14x14, batch 8, bf16
      // 8.8 us, a channel at a time 10.5; 260 -> 256 of 56x56, batch 128, f16 37.0 and 33.6; float32 384 -> 256 of 14x14, one image 10.4 and
      // 12.2; 512 -> 256 of 33x33, batch 32 26.4 and 23.7, all channels at once 21.8.
      int col[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int w = w0 + e * step_w;
        col[e] = w < 0 ? 0 : w < p.w_in ? w : p.w_in - 1;
      }
      auto line = [&](int c) { return src + (o0 - w0 + (c < nch ? c * plane : 0)); };
      if (!UNIT && gridDim.x - p.w_blocks <= (W == 8 ? 64u : 128u)) {
        bool any[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) any[e] = __builtin_amdgcn_ballot_w64(in_row(e)) != 0;
        uint32_t t[8][8];                           // (a half in a word of its own until all are there)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const E* at = line(c);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            t[c][e] = 0;
            if (any[e]) {
              const E v = at[col[e]];
              t[c][e] = W == 8 ? __builtin_bit_cast(uint32_t, (float)v) : (uint32_t)v;
            }
          }
        }
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
          for (int e = 0; e < 8; ++e) asm("" : "+v"(t[c][e]));
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
          for (int i = 0; i < W; ++i) raw[c][i] = W == 8 ? t[c][i] : t[c][2 * i & 7] | t[c][(2 * i + 1) & 7] << 16;
      } else if constexpr (!UNIT && W == 8) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const E* at = line(c);
#pragma unroll
          for (int e = 0; e < 8; ++e) raw[c][e] = __builtin_bit_cast(uint32_t, (float)at[col[e]]);
          __builtin_amdgcn_sched_barrier(0);        // (addresses of later channels not before: 184 registers)
        }
      } else {
#pragma unroll 1
        for (int c = 0; c < nch; ++c) {
          const E* at = line(c);
          E t[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] = at[col[e]];
          uint32_t u[W];
          __builtin_memcpy(u, t, sizeof u);
#pragma unroll
          for (int x = 0; x < 8; ++x)
#pragma unroll
            for (int i = 0; i < W; ++i) raw[x][i] = x == c ? u[i] : raw[x][i];
        }
      }
      clear(eight);
    }
  }
#pragma unroll
  for (int c = 0; c < 8; ++c)
#pragma unroll
    for (int i = 0; i < W; ++i) asm("" : "+v"(raw[c][i]));      // words, not halves, cross the branches
  E in[8][8];
  __builtin_memcpy(in, raw, sizeof in);
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
