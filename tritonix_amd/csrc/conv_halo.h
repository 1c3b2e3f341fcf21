// conv2d forward with the input window of a tile resident in LDS (16-bit types).
//
// out[c_out, pixel] = sum over (channel block, filter tap, channel) of W * X: a workgroup owns BM output channels and BN
// consecutive output pixels.  Of 32 input channels at a time it holds every input row those pixels need -- the halo included,
// padding written out as zeros -- as [row][column][channel], and takes all filter taps from there: a tap is a constant added to
// an LDS address.  Against the packed route (conv_pack.h) the pass that copies the whole input to [pixel][channel] falls away, and an
// input element crosses from the L2 to the LDS once per channel block instead of once per tap; only the weight, laid out as
// [c_out][channel block][tap][32 channels] by a small launch before this one (halo_weight_kernel), goes through a DMA ring.
//
// The K loop runs over k steps of 32 (a channel block's taps, then the next block's), KSP of them between two barriers.  In a
// period that starts with the next block's window due, each wave first puts what it fetched one block earlier into the other window
// buffer (eight 16-byte row pieces of eight channels: an 8x8 transpose by byte permutes, one 16-byte store per pixel), spread over
// the MFMA slots, and fetches the following block's at the period's end.  The order matters: the compiler waits for a fetched
// register by counting its own loads only, so between a fetch and its use it would wait for every ring load issued in between; at a
// period's start there is none.
#pragma once
#include "gemm_tile.h"

namespace tnx {

struct HaloGeom {
  const uint8_t* x;
  int c_in, h_in, w_in, plane;     // plane: h_in * w_in
  int batch, x_elems;
  int width;                       // pixels of a tile: BN, or less where that makes them whole output rows
  int rows_img;                    // rows of one image with its padding, as far as any output needs them
  int stride_h, stride_w, pad_h, pad_w;
  int fh, fw, dil_h, dil_w, taps;
  int cps, rowslots;               // columns of one parity (stride_w == 2: even and odd ones lie apart), pixel slots per window row
  int hw_out, hwp, w_out;          // output plane, the same rounded up to 8, output row
  int cpr;                         // chunks of 8 columns per input row
  int rows;                        // of the largest window
  int buf_bytes;                   // one window buffer
  int blocks, ksteps;              // blocks of 32 channels; blocks * taps
  FastDiv div_img, div_hwp, div_w, div_cpr, div_taps, div_fw;
};

// A pixel slot: 32 channels in four 16-byte chunks.  The 16 lanes that a fragment read serves in one cycle ({0-3, 12-15, 20-27}) are
// eight slots with chunk kg and the eight between them with kg + 1.  At 96 bytes from slot to slot the first eight fall on the even
// chunks of a bank row and the others on the odd ones, wherever a filter tap makes them start.  At 64 bytes the chunk index is
// XOR-ed with a bit of the slot to the same effect, but the tap then changes the XOR: four vector instructions a read
// instead of one, for two thirds of the LDS (what a stride of 2 needs, whose windows have four times the pixels of their outputs).
template <int SLOT> __device__ __forceinline__ uint32_t halo_at(uint32_t slot_bytes, uint32_t chunk16) {
  return SLOT == 64 ? slot_bytes + (chunk16 ^ ((slot_bytes >> 3) & 0x20u)) : slot_bytes + chunk16;
}

// Byte of channel c of block cb where the first channel's is `src`; and the first channel's of a lane that has no row: the tensor's end,
// so that every channel's stays past it, where the range check drops the load.  (Not the largest number: with what the channels add it
// wraps to a place inside the tensor.  The tensor's end does where it and an image make 4 GiB; what is read then goes to the spill place.)
__host__ __device__ constexpr uint32_t halo_channel_at(uint32_t src, int cb, int c, int plane) {
  return src + (uint32_t)(cb * 32 + c) * 2u * (uint32_t)plane;
}
__host__ __device__ constexpr uint32_t halo_nowhere(uint32_t x_bytes) { return x_bytes; }
constexpr bool halo_nowhere_holds(uint32_t x_bytes, int c_in, int plane) {
  for (int c = 0; c < (c_in + 31) / 32 * 32; ++c)
    if (halo_channel_at(halo_nowhere(x_bytes), c / 32, c % 32, plane) < x_bytes) return false;
  return true;
}
static_assert(halo_nowhere_holds(32u * 128 * 3136 * 2, 128, 3136) && halo_nowhere_holds(17u * 3 * 5 * 2, 17, 15) &&
              halo_nowhere_holds(2u * 900 * 1048576 * 2, 900, 131072), "lanes without a row read nothing");

// Behind the windows: an offset per k step, of one period past the end too, and from the next 16-byte boundary on a place per lane.
__host__ __device__ constexpr int halo_table_bytes(int ksp, int periods) { return (ksp * (periods + 1) * 4 + 15) / 16 * 16; }
constexpr int HALO_SPILL_BYTES = 64 * 16;

// BM output channels x BN pixels, 8 waves; the ring holds R periods of KSP k steps
template <class T, int BM, int BN, int KSP_, int R_, int SLOT_> struct HaloCfg {
  typedef TileCfg<T, BM, BN, 64, 8, 2> C;
  static constexpr int KSP = KSP_, R = R_, SLOT = SLOT_, NSUB = KSP / 2;
  static_assert(SLOT == 64 || SLOT == 96, "pitches whose fragment reads are free of bank conflicts");
  static constexpr int PERIOD_BYTES = NSUB * C::A_BYTES, RING_BYTES = R * PERIOD_BYTES;
  static constexpr int LPW = PERIOD_BYTES / 1024 / 8;              // ring loads of a wave per period
  static_assert(KSP % 2 == 0 && PERIOD_BYTES % 8192 == 0 && C::BK == 64 && C::ES == 2 && C::MI == 16, "slabs of two k steps, whole loads");
};

template <class T, class H>
__global__ __launch_bounds__(512, 2) void conv_halo_kernel(GemmParams p, HaloGeom h) {
  typedef typename H::C C;
  constexpr int BM = C::BM, BN = C::BN, NW = C::NW, TM = C::TM, TN = C::TN, MI = C::MI, KSP = H::KSP, R = H::R, LPW = H::LPW, SLOT = H::SLOT;
  constexpr int NMMA = TM * TN;
  typedef Mma<T, MI> MMA;
  typedef typename MMA::acc_t acc_t;
  extern __shared__ __attribute__((aligned(1024))) uint8_t halo_smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(uint8_t __attribute__((address_space(3)))*)halo_smem;
  const uint32_t win0 = lds0 + H::RING_BYTES;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int pid_m, pid_n;
  swizzle2d(xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n, 8), p, &pid_m, &pid_n);
  const int m0 = pid_m * BM, n0 = pid_n * h.width, n1 = n0 + h.width < p.cv.n_total ? n0 + h.width : p.cv.n_total;
  const int KT = (h.ksteps + KSP - 1) / KSP;              // periods; at least two (the host sees to it)

  // ---- output pixels -> window rows.  Rows are counted through all images, `rows_img` each.
  auto place = [&](int n, int* row, int* col) __attribute__((always_inline)) {
    n = n < n1 ? n : n1 - 1;                              // pixels past the tile's end are computed and dropped
    const int img = (int)fd_div((uint32_t)n, h.div_hwp);
    int r = n - img * h.hwp;
    r = r < h.hw_out ? r : h.hw_out - 1;
    const int ho = (int)fd_div((uint32_t)r, h.div_w);
    *row = img * h.rows_img + ho * h.stride_h;
    *col = r - ho * h.w_out;
  };
  int row0, rowl, unused;
  place(n0, &row0, &unused);
  place(n1 - 1, &rowl, &unused);
  row0 = __builtin_amdgcn_readfirstlane(row0);
  const int rows = __builtin_amdgcn_readfirstlane(rowl) - row0 + (h.fh - 1) * h.dil_h + 1;

  const int wy = wave / C::WGN, wx = wave % C::WGN;
  uint32_t b_base[TN];                                    // window byte of the lane's pixel of each fragment, at tap (0, 0)
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    int r, c;
    place(n0 + wx * C::WTN + j * MI + (lane & 15), &r, &c);
    b_base[j] = win0 + (uint32_t)((r - row0) * h.rowslots + c) * SLOT + (SLOT == 64 ? 0u : (uint32_t)(lane >> 4) * 16u);
  }

  // ---- the weight ring
  const uint8_t* a_sbase = uniform_ptr(p.a + (int64_t)m0 * p.sam * 2);
  uint32_t a_voff[LPW];
  const int mrem = (int)p.m - 1 - m0;
#pragma unroll
  for (int q = 0; q < LPW; ++q) {
    const int P = (q * NW + wave) * 64 + lane, sub = P / (BM * 8), row = P / 8 % BM, c = (P % 8) ^ C::swzA(row);
    a_voff[q] = (uint32_t)(row < mrem ? row : mrem) * (uint32_t)(p.sam * 2) + (uint32_t)(sub * 128 + c * 16);
  }
  auto ring_op = [&](int q, uint32_t slot) __attribute__((always_inline)) {
    dma16(a_sbase, a_voff[q], slot + (uint32_t)(q * NW + wave) * 1024u);
  };

  // ---- the window.  A thread moves 8 channels x 8 columns of one row, the same ones of every channel block; four neighbouring lanes
  // take neighbouring chunks (64 bytes of a plane where rows are whole chunks), four such groups the four groups of 8 channels: the
  // loads want neighbours along a row, but those are stored 8 slots apart, on the same banks.  (512 x 512 channels, 3x3 on 14x14, batch
  // 32: with sixteen neighbours along a row 45.5 us, with four 43.0; with every other pair's halves exchanged, so that two lanes
  // meet on a bank instead of four, 44.1: the exchange costs more than it saves.)
  const uint32_t x_bytes = (uint32_t)h.x_elems * 2u;
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(h.x), 0, x_bytes, 0x00020000);
  const int cg8 = (tid >> 2 & 3) * 8;
  uint32_t t_src;                                         // byte of (first channel, first column) in block 0, or past the tensor
  uint32_t t_lds;                                         // window byte of the first column
  int t_cols;                                             // columns that belong to the row
  {
    const int c = (tid >> 4) * 4 + (tid & 3), pr = (int)fd_div((uint32_t)c, h.div_cpr), w0 = (c - pr * h.cpr) * 8;
    const int g = row0 + pr, img = (int)fd_div((uint32_t)g, h.div_img), ih = g - img * h.rows_img - h.pad_h;
    const bool ok = pr < rows && img < h.batch && (uint32_t)ih < (uint32_t)h.h_in;
    t_src = ok ? ((uint32_t)(img * h.c_in + cg8) * (uint32_t)h.plane + (uint32_t)(ih * h.w_in + w0)) * 2u : halo_nowhere(x_bytes);
    const int pc = w0 + h.pad_w, left = h.w_in - w0, used = h.rowslots - pc;
    t_cols = !ok ? 0 : left < used ? left : used;
    t_lds = win0 + (uint32_t)(pr * h.rowslots + (h.stride_w == 2 ? pc >> 1 : pc)) * SLOT;
  }
  const uint32_t table = win0 + 2u * (uint32_t)h.buf_bytes, spill = table + (uint32_t)halo_table_bytes(KSP, KT) + (uint32_t)lane * 16u;
  const bool has_rows = wave * 16 < rows * h.cpr;         // this wave moves anything at all
  i32x4 v[8];
  auto fetch_one = [&](int c, int cb) __attribute__((always_inline)) {
    // (channels past the last one: zeros past the tensor, or whatever is there before its end, cleared by `put_begin`)
    v[c] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, halo_channel_at(t_src, cb, c, h.plane), 0, 0);
  };
  // even and odd columns of a chunk: neighbours, or apart where the stride is 2
  const bool strided = h.stride_w == 2, odd0 = strided && (h.pad_w & 1);
  const uint32_t apart = strided ? (uint32_t)h.cps * SLOT : (uint32_t)SLOT;
  const uint32_t even_off = odd0 ? apart : 0u, odd_off = odd0 ? (uint32_t)SLOT : apart;
  const uint32_t col_step = strided ? SLOT : 2 * SLOT;
  auto put_begin = [&](int cb) __attribute__((always_inline)) {
    if (cb != h.blocks - 1) return;
    const int nch = h.c_in - cb * 32 - cg8;               // channels of this group that exist
    // the tensor's last chunk may end past it, and the loads drop every dword that is not whole: element by element
    const uint32_t last = halo_channel_at(t_src, cb, nch - 1, h.plane);
    const bool over = t_cols > 0 && nch > 0 && nch <= 8 && last + 16u > x_bytes;
    if (__builtin_amdgcn_ballot_w64(over) != 0) {
      uint16_t e[8];
#pragma unroll
      for (int x = 0; x < 8; ++x) e[x] = over && last + 2 * x < x_bytes ? *(const uint16_t*)(h.x + last + 2 * x) : (uint16_t)0;
      i32x4 w;
      __builtin_memcpy(&w, e, 16);
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = over && c == nch - 1 ? w : v[c];
    }
    if (h.c_in & 31) {
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = c < nch ? v[c] : i32x4{0, 0, 0, 0};
    }
  };
  auto put_one = [&](int e, uint32_t buf) __attribute__((always_inline)) {
    i32x4 o;
#pragma unroll
    for (int d = 0; d < 4; ++d)
      o[d] = (int)__builtin_amdgcn_perm((uint32_t)v[2 * d + 1][e / 2], (uint32_t)v[2 * d][e / 2], e & 1 ? 0x07060302u : 0x05040100u);
    // (columns that are not the row's go to a place of the lane's own behind the table: cheaper than masking lanes)
    const uint32_t at = halo_at<SLOT>(t_lds + (buf + (e & 1 ? odd_off : even_off) + (e / 2) * col_step), (uint32_t)cg8 * 2u);
    *TNX_LDS(i32x4, e < t_cols ? at : spill) = o;
  };

  // ---- prologue: ring and first channel block under way, windows cleared (what no input covers stays zero for good)
#pragma unroll
  for (int s = 0; s < R; ++s)
    if (s < KT) {
#pragma unroll
      for (int q = 0; q < LPW; ++q) ring_op(q, lds0 + s * H::PERIOD_BYTES);
      a_sbase += KSP * 64;
    }
  if (has_rows) {
#pragma unroll
    for (int c = 0; c < 8; ++c) fetch_one(c, 0);
  }
  for (int at = tid * 16; at < 2 * h.buf_bytes; at += 512 * 16) *TNX_LDS(i32x4, win0 + at) = i32x4{0, 0, 0, 0};
  // window offset of every k step: its channel block's buffer and its filter tap
  for (int q = tid; q < KSP * (KT + 1); q += 512) {
    const int cb = (int)fd_div((uint32_t)q, h.div_taps), r = q - cb * h.taps, th = (int)fd_div((uint32_t)r, h.div_fw);
    const int dw = (r - th * h.fw) * h.dil_w;
    const int slot = th * h.dil_h * h.rowslots + (strided ? (dw & 1) * h.cps + (dw >> 1) : dw);
    *TNX_LDS(uint32_t, table + q * 4) = (uint32_t)(slot * SLOT + (cb & 1) * h.buf_bytes);
  }
  __syncthreads();
  if (has_rows) {
    put_begin(0);
#pragma unroll
    for (int e = 0; e < 8; ++e) put_one(e, 0u);
    if (h.blocks > 1) {
#pragma unroll
      for (int c = 0; c < 8; ++c) fetch_one(c, 1);
    }
  }
  // Block cb's window is put in period cb * taps / KSP - 2, the one before its first read: by then the last read of the block two
  // before it, (cb - 1) * taps - 1, lies behind a barrier (taps >= 2 * KSP).
  int ev_cb = 1;
  auto due = [&]() __attribute__((always_inline)) { return ev_cb < h.blocks ? ev_cb * h.taps / KSP - 2 : 0x7fffffff; };
  int ev_due = has_rows ? due() : 0x7fffffff;

  // ---- fragments: two register sets of the window's and of the weight's -- or, in the tiles that need the registers, one set of the
  // weight's but for the last row-block: row i's is read anew once its MFMAs are issued
  constexpr bool ONE_A = TM * TN * 4 > 80;
  const int a_row = wy * C::WTM + (lane & 15);
  const uint32_t a_off = (uint32_t)(a_row * 128 + (((lane >> 4) ^ C::swzA(a_row)) << 4));
  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{};
  i32x4 fa[2][TM], fb[2][TN];
  auto a_set = [](int set, int i) { return ONE_A && i + 1 < TM ? 0 : set; };
  uint32_t taps_at = table;
  i32x4 tap = {0, 0, 0, 0};
  auto next_taps = [&]() __attribute__((always_inline)) {
    if constexpr (KSP == 4) {
      tap = *TNX_LDS(i32x4, taps_at);
    } else {
      const i32x2 t = *TNX_LDS(i32x2, taps_at);
      tap = i32x4{t.x, t.y, 0, 0};
    }
    taps_at += KSP * 4;
  };
  auto read_b = [&](int set, int j, int ks) __attribute__((always_inline)) { fb[set][j] = *TNX_LDS(i32x4, halo_at<SLOT>(b_base[j] + (uint32_t)tap[ks], SLOT == 64 ? (uint32_t)(lane >> 4) * 16u : 0u)); };
  auto read_a = [&](int set, int i, int ks, uint32_t slab) __attribute__((always_inline)) {
    fa[a_set(set, i)][i] = *TNX_LDS(i32x4, ((slab + (ks >> 1) * C::A_BYTES + a_off) ^ ((ks & 1) * 64)) + i * MI * 128);
  };
  auto mma_one = [&](int set, int x) __attribute__((always_inline)) {
    const int i = x / TN;
    int j = x % TN;
    if (i & 1) j = TN - 1 - j;
    acc[i][j] = MMA::run(fb[set][j], fa[a_set(set, i)][i], acc[i][j]);
  };
  // One k step's MFMAs with the reads of k step `ks` (of the period-slab at `slab`) behind them, and extra(x) in slot x
  auto step = [&](int ks, uint32_t slab, auto extra) __attribute__((always_inline)) {
    const int set = ks & 1, mset = set ^ 1;
    constexpr int RPM = (TN + TM + NMMA - 1) / NMMA;
    int rd = 0;
#pragma unroll
    for (int x = 0; x < NMMA; ++x) {
      mma_one(mset, x);
      if constexpr (ONE_A) {
        if (x < TN) read_b(set, x, ks);
        if (x == TN) read_a(set, TM - 1, ks, slab);
        if (x % TN == TN - 1 && x / TN + 1 < TM) read_a(set, x / TN, ks, slab);
      } else {
#pragma unroll
        for (int r = 0; r < RPM; ++r) {
          if (rd < TN) read_b(set, rd, ks);
          else if (rd < TN + TM) read_a(set, rd - TN, ks, slab);
          ++rd;
        }
      }
      extra(x);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto nothing = [](int) {};

  if (has_rows && h.blocks > 1) { TNX_WAIT_VM(8); } else { TNX_WAIT_VM(0); }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  next_taps();
#pragma unroll
  for (int j = 0; j < TN; ++j) read_b(0, j, 0);
#pragma unroll
  for (int i = 0; i < TM; ++i) read_a(0, i, 0, lds0);
#pragma unroll
  for (int s = 1; s < KSP; ++s) step(s, lds0, nothing);
  next_taps();

  uint32_t freed = lds0, next = lds0 + H::PERIOD_BYTES;
  bool fetched = false;                                   // the youngest eight loads of this wave are a fetch
  bool loaded = R > 2 && KT > 2;                          // ... and before them, the ring loads of the period-slab after the next
  int t = 0;
  // One period: the MFMAs of period-slab t's last k step and of period-slab t + 1's others, the reads of all of period-slab t + 1.
  auto period = [&](auto with_event) __attribute__((always_inline)) {
    constexpr bool EVENT = decltype(with_event)::value;
    // period-slab t + 1 has landed; nobody reads slab t any more, nor the windows of blocks before the present one
    if (R > 2 && loaded) {
      if (fetched) { TNX_WAIT_VM((R > 2 ? LPW : 0) + 8); } else { TNX_WAIT_VM(R > 2 ? LPW : 0); }
    } else {
      if (fetched) { TNX_WAIT_VM(8); } else { TNX_WAIT_VM(0); }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const bool load = t + R < KT;
    // slots of the first step (or two): the window's eight columns, and the ring's loads
    constexpr int SPLIT = KSP > 2 && NMMA < 16 ? 2 : 1, PUTS = 8 / SPLIT;
    const uint32_t buf = (uint32_t)((ev_cb & 1) * h.buf_bytes);
    const bool more = EVENT && ev_cb + 1 < h.blocks;
    if constexpr (EVENT) {
      TNX_WAIT_VM(0);                // what was fetched is there: said here, once, the compiler does not wait behind the ring's loads
      put_begin(ev_cb);
    }
#pragma unroll
    for (int s = 0; s < KSP; ++s) {
      step(s, next, [&](int x) __attribute__((always_inline)) {
        if (EVENT && s < SPLIT) {
          const int lo = s * PUTS + x * PUTS / NMMA, hi = s * PUTS + (x + 1) * PUTS / NMMA;
#pragma unroll
          for (int e = lo; e < hi; ++e) put_one(e, buf);
        }
        if (s == 0) {
          const int lo = x * LPW / NMMA, hi = (x + 1) * LPW / NMMA;
          if (hi > lo && load) {
#pragma unroll
            for (int q = lo; q < hi; ++q) ring_op(q, freed);
          }
        }
        if (EVENT && s == KSP - 1) {
          const int lo = x * 8 / NMMA, hi = (x + 1) * 8 / NMMA;
          if (hi > lo && more) {
#pragma unroll
            for (int c = lo; c < hi; ++c) fetch_one(c, ev_cb + 1);
          }
        }
      });
    }
    next_taps();
    fetched = more;
    if (load) a_sbase += KSP * 64;
    loaded = load;
    freed = next;
    next = next + H::PERIOD_BYTES == win0 ? lds0 : next + H::PERIOD_BYTES;
    ++t;
  };
  // (one loop around both kinds of period, not a branch between two kinds inside one: accumulators that come out of two branches
  // are copied where they meet, 400 spilled registers)
  for (;;) {
    const int stop = ev_due < KT - 2 ? ev_due : KT - 2;
    while (t < stop) period(BoolTag<false>{});
    if (t >= KT - 2) break;
    period(BoolTag<true>{});
    ++ev_cb;
    ev_due = due();
  }
  // the last period-slab, which may hold fewer k steps than KSP
  const int rem = h.ksteps - (KT - 1) * KSP;
  TNX_WAIT_VM(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < KSP; ++s)
    if (s <= rem) step(s, next, nothing);
  if (rem == KSP) {
#pragma unroll
    for (int x = 0; x < NMMA; ++x) mma_one(1, x);
  }

  // ---- epilogue: the strips are laid over ring and windows
  __syncthreads();
  const uint32_t strip = lds0 + wave * EpiStage<C>::WAVE_BYTES;
  p.cv.n_total = n1;
  if (p.out_dtype == DT_F32) epilogue_store_conv<T, C, OutF32>(acc, p.c, strip, lane, m0 + wy * C::WTM, n0 + wx * C::WTN, p.cv);
  else epilogue_store_conv<T, C, typename OutOf<T>::type>(acc, p.c, strip, lane, m0 + wy * C::WTM, n0 + wx * C::WTN, p.cv);
}

typedef hipError_t (*halo_launch_fn)(const GemmParams& p, const HaloGeom& h, unsigned grid, int lds_bytes, hipStream_t stream);
struct HaloEntry {
  int dtype, bm, bn, ksp, ring, slot;    // k steps of a period, periods in the ring, bytes of a pixel slot
  int ring_bytes, strip_bytes;     // LDS of the weight ring and of the epilogue that takes its place
  halo_launch_fn launch;
};
template <class T, class H>
hipError_t launch_halo(const GemmParams& p, const HaloGeom& h, unsigned grid, int lds_bytes, hipStream_t stream) {
  GemmParams q = p;
  set_order_divisors(&q);
  hipLaunchKernelGGL((conv_halo_kernel<T, H>), dim3(grid), dim3(512), lds_bytes, stream, q, h);
  return hipGetLastError();
}
#define TNX_HALO_ENTRY(TAG, BM, BN, KSP, R, SLOT)                                                                           \
  {TAG::ID, BM, BN, KSP, R, SLOT, HaloCfg<TAG, BM, BN, KSP, R, SLOT>::RING_BYTES, EpiStage<HaloCfg<TAG, BM, BN, KSP, R, SLOT>::C>::BYTES, \
   &launch_halo<TAG, HaloCfg<TAG, BM, BN, KSP, R, SLOT>>}

// The weight as that kernel reads it: [c_out][channel block][tap][32 channels], rows zero-filled to whole periods.  A thread takes the
// taps of 8 channels of one output channel, which lie in one run: TAPS 16-byte loads, 16-byte stores, byte permutes between them.
// Bound by latency and by the lines a wave's loads touch, so a workgroup is one wave and the CUs share them: 256 x 256 x 3x3
// 3.0 us a launch, in workgroups of four waves 6.1; 512 x 512 5.2; 128 x 128 2.2.  (Done by the tile kernel's own first workgroups while the
// others wait at flags it takes as long: 128 channels of 56x56, stride 2, batch 32, 17.2 us against 17.1 -- and 20.4 with what
// clearing the flags behind it costs.)
struct HaloWeight {
  const uint8_t* w;
  uint8_t* out;
  int c_in, c_out, groups, chunks;   // groups of 8 channels, padded to whole blocks; 16-byte chunks of a row
  int taps;
  FastDiv div_groups;
};
template <int TAPS> __global__ __launch_bounds__(64) void halo_weight_kernel(HaloWeight p) {
  const int id = blockIdx.x * 64 + threadIdx.x, taps = TAPS ? TAPS : p.taps;
  const int co = (int)fd_div((uint32_t)id, p.div_groups), cg = id - co * p.groups;
  if (co >= p.c_out) return;
  const uint16_t* src = (const uint16_t*)p.w + ((int64_t)co * p.c_in + cg * 8) * taps;
  i32x4* row = (i32x4*)p.out + (int64_t)co * p.chunks;
  i32x4* dst = row + (cg >> 2) * taps * 4 + (cg & 3);
  const int nch = p.c_in - cg * 8;
  if (TAPS && nch >= 8) {
    uint16_t e[TAPS ? TAPS * 8 : 1];
#pragma unroll
    for (int x = 0; x < TAPS; ++x) {
      const i32x4 v = *(const i32x4_loose*)(src + x * 8);
      __builtin_memcpy(e + x * 8, &v, 16);
    }
#pragma unroll
    for (int t = 0; t < TAPS; ++t) {
      uint16_t o[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) o[c] = e[c * TAPS + t];
      i32x4 v;
      __builtin_memcpy(&v, o, 16);
      dst[t * 4] = v;
    }
  } else {
#pragma unroll 1
    for (int t = 0; t < taps; ++t) {
      uint16_t o[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) o[c] = c < nch ? src[c * taps + t] : (uint16_t)0;
      i32x4 v;
      __builtin_memcpy(&v, o, 16);
      dst[t * 4] = v;
    }
  }
  // behind the last block: the k steps that fill its period
  if (cg >= p.groups - 4)
    for (int x = p.groups * taps + (cg & 3); x < p.chunks; x += 4) row[x] = i32x4{0, 0, 0, 0};
}

}  // namespace tnx
