// The inner loop of products in LDS tiles (gfx950), bf16 or e4m3: x and w come
// in chunks of 128 bytes of a row, from memory to LDS directly, into a ring.
//
// The operands of a step are read from LDS before the products of the step
// before, and the first ones of a stage before the last products of the stage
// before it, so that no product waits for a read.  What bounds it then: 256 x
// 256 tiles the power that products may take (a product of 8192 x 28672 x 4096
// without its loads 1325 us with random numbers, 1060 with zeros), smaller ones
// the bytes in flight.  Four prompts of 500 tokens through 4 layers of 8 experts
// of 14336 x 4096 5645 -> 5435 us, a prompt of 512 through 8 dense layers 2265 ->
// 2240, where every step waited for its own reads.
#pragma once

#include "common.h"

// Rows in memory from `base` on: 16 bytes a lane, of byte offset `at` (below
// 4 GB) + `from`, which is uniform, to LDS address l + lane * 16.  Loads by a
// buffer's address, for the compiler takes those by a global one for flat ones,
// and then waits for all LDS reads where it needs the oldest.
//
// ONCE (non-temporal): rows that no other workgroup reads, or few at the same
// time, as weights.  A load that waits for memory otherwise holds a line of the
// unit's cache, of which there are 256, and answers come in order: a unit gets 47
// GB/s from memory and with this 87, all of them 6.2 TB/s and 7.3.  What is read
// again, as x by the tiles of all outputs, is slower with it.  us: 64 rows of 28672
// x 4096 41.4 -> 38.4, 1 of 4096 x 14336 in 4 parts 21.8 -> 19.7, 256 of 28672 x
// 4096 74 -> 66, 512 of 4096 x 14336 64 -> 61; weights that the memory's cache of
// 256 MB has from the last time, which a model's layers together leave no room
// for, 0 to 20 % slower.
enum { ONCE = 2 };
struct RowLoads {
  __amdgpu_buffer_rsrc_t rows;
  DEV explicit RowLoads(const void* base)
      : rows(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0,
                                               0xffffffff, 0x00020000)) {}
  template <int AUX = 0>
  DEV void to_lds(char* l, unsigned at, unsigned from) const {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rows, (__attribute__((address_space(3))) unsigned*)l, 16, at, from, 0,
        AUX);
  }
};

// 16-byte unit c of row r of a chunk in LDS.  16 lanes read at a time, 16 rows
// of one unit, and two rows fill the 64 banks: so the unit turns with every
// second row.
DEV int chunk_unit(int r, int c) { return r * 128 + ((c ^ (r >> 1 & 7)) << 4); }

typedef __attribute__((ext_vector_type(8))) int int32x8_t;

// BM rows of x, BN of w; WM * WN waves have BM / WM by BN / WN.  A stage has KC
// chunks: BM rows of x, then BN of w, of each.
//
// SPREAD: a stage's loads are issued between the products of the next one, not
// all behind the barrier that frees its slot, where 48 KB take a compute unit's
// memory pipe some 770 cycles and no wave that waits to issue its own gets to a
// product.  They have one stage less to arrive in, so it takes three.  us, with
// weights from memory: 512 rows of 4096 x 14336 in 4 parts 66 -> 62, of 6144 x
// 4096 in 2 36.1 -> 34.0, 256 of 28672 x 4096 75 -> 70.  128 x 128 tiles, which
// have less to issue, are even (256 rows of 4096 x 14336 45.1 45.5), smaller ones
// slower (32 of 2048 x 7168 8.3 8.9).
template <int BM, int BN, int WM, int WN, int STAGES, int KC, bool FP8>
struct TileLoop {
  static constexpr int WAVES = WM * WN;
  static constexpr int NI = BN / WN / 32, MI = BM / WM / 32;
  static constexpr int LX = BM / 8 / WAVES, LW = BN / 8 / WAVES;  // a chunk
  static constexpr int SUB = (BM + BN) * 128, STAGE = SUB * KC;
  static constexpr int BYTES = STAGES * STAGE;
  static constexpr int LOADS = (LX + LW) * KC;
  // A product takes 16 bytes a lane of a row, of e4m3 32: 64 columns in twice
  // the time of 16.  64 rows of 3072 x 2048 7.4 -> 6.4 us, 1 of 6144 x 4096 11.5
  // -> 10.6.  Against 64 bits both are off by 1.3e-5 of the result, with
  // magnitudes that differ by e^3 3.8e-5.
  static constexpr int UNITS = FP8 ? 2 : 1, STEPS = 4 / UNITS * KC;
  static_assert(LX * WAVES * 8 == BM && LW * WAVES * 8 == BN, "loads");
  static_assert((STAGES - 1) * LOADS < 64, "the counter of loads");

  struct Frag {
    short8_t x[MI][UNITS], w[NI][UNITS];
  };
  f32x16_t acc[NI][MI];

  DEV void read(Frag& f, const char* base, int x_at, int w_at, int step) {
    #pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int unit = step * UNITS + u, k = unit & 3;
      const char* p = base + (unit >> 2) * SUB;
      #pragma unroll
      for (int n = 0; n < NI; ++n)
        f.w[n][u] = *reinterpret_cast<const short8_t*>(
            p + (w_at ^ k << 5) + n * 32 * 128);
      #pragma unroll
      for (int m = 0; m < MI; ++m)
        f.x[m][u] = *reinterpret_cast<const short8_t*>(
            p + (x_at ^ k << 5) + m * 32 * 128);
    }
  }
  DEV void products(const Frag& f) {
    #pragma unroll
    for (int n = 0; n < NI; ++n)
      #pragma unroll
      for (int m = 0; m < MI; ++m)
        if constexpr (FP8) {
          union { short8_t s[2]; int32x8_t v; } u{{f.w[n][0], f.w[n][1]}},
              v{{f.x[m][0], f.x[m][1]}};
          acc[n][m] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
              u.v, v.v, acc[n][m], 0, 0, 0, 0, 0, 0);    // e4m3, no scales
        } else {
          acc[n][m] = mfma32(f.w[n][0], f.x[m][0], acc[n][m]);
        }
  }

  static constexpr bool SPREAD = BM == 256 && STAGES > 2;

  // stage(slot, d, i) issues load i of this wave's LOADS of stage d of the ring.
  // Every wave has to call this; those that are not live only load.
  template <class Stage>
  DEV void run(char* lds, int wm, int wn, int stages, bool live,
               Stage stage) {
    const int lane = threadIdx.x & 63, col = lane & 31, hf = lane >> 5;
    const int x_at = chunk_unit(wm * MI * 32 + col, hf);
    const int w_at = BM * 128 + chunk_unit(wn * NI * 32 + col, hf);
    auto loads = [&](int slot, int d, int from, int to) {
      #pragma unroll
      for (int i = 0; i < LOADS; ++i)
        if (i >= from && i < to) stage(slot, d, i);
    };
    #pragma unroll
    for (int n = 0; n < NI; ++n)
      #pragma unroll
      for (int m = 0; m < MI; ++m) acc[n][m] = f32x16_t(0.f);
    #pragma unroll
    for (int d = 0; d < STAGES; ++d)
      if (d < stages) loads(d, d, 0, LOADS);
    if (stages >= STAGES)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier"
                   ::"n"((STAGES - 1) * LOADS) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    Frag f[2];
    if (live) read(f[0], lds, x_at, w_at, 0);
    int slot = 0;
    for (int d = 0; d < stages; ++d) {
      const char* base = lds + slot * STAGE;
      // SPREAD: the slot of stage d - 1
      const int last = slot == 0 ? STAGES - 1 : slot - 1;
      const bool more = SPREAD && d > 0 && d - 1 + STAGES < stages;
      if (SPREAD || live) {
        #pragma unroll
        for (int k = 0; k < STEPS - 1; ++k) {
          if (live) read(f[(k + 1) & 1], base, x_at, w_at, k + 1);
          if (more)
            loads(last, d - 1 + STAGES, LOADS * k / (STEPS - 1),
                  LOADS * (k + 1) / (STEPS - 1));
          if (live) {
            __builtin_amdgcn_sched_barrier(0);
            products(f[k & 1]);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      const int next = slot == STAGES - 1 ? 0 : slot + 1;
      if (d + 1 < stages) {
        // stage d + 1 has landed and all of d has been read, by every wave:
        // its slot is free
        if (d + STAGES <= stages)
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                       ::"n"((STAGES - 2) * LOADS) : "memory");
        else
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier"
                       ::: "memory");
        if (live) read(f[0], lds + next * STAGE, x_at, w_at, 0);
        if (!SPREAD && d + STAGES < stages) loads(slot, d + STAGES, 0, LOADS);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (live) products(f[1]);
      slot = next;
    }
    // The last sums are there before anything reads them.  The compiler's own
    // wait is not there on every way out of the loop: where the first reads were
    // copies from accumulation registers in a block of their own, the second one
    // came 6 instructions after the products, which take 11.  As operands before
    // and after it the sums can pass this wait in neither direction; in vector
    // registers (two waves a SIMD or more) there are no copies.
    in_order();
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
    in_order();
  }
  DEV void in_order() {
    #pragma unroll
    for (int n = 0; n < NI; ++n)
      #pragma unroll
      for (int m = 0; m < MI; ++m) asm volatile("" : "+v"(acc[n][m]));
  }
};

// The loop of tiles as wide as registers allow, 8 waves.  A wave has MB blocks of B
// rows of x and NB of w, and loads LX and LW times 8 rows of a chunk.  bf16 takes 16 x
// 16 x 32 products, e4m3 32 x 32 x 64: a chunk is two steps of 64 bytes.
//
// 256 x 256 tiles have room for two stages, in which a chunk has less time to arrive
// than memory needs; so x and w have slots apart, w, which comes from farther away,
// always three, x three (XS) where they fit.  Reads of the next step and loads are
// issued one by one between a step's products, and not all at once.
//
// What bounds it is power, and then the bytes on their way: 256 x 256 tiles of 2000
// rows of 28672 x 4096 an expert without loads 2670 us with 32 x 32 products, 2390 with
// 16 x 16 ones, which read and write half the sums; without products 2590 with two
// stages, 1970 with slots apart.
template <int BM, int BN, int MB, int NB, int LX, int LW, bool FP8>
struct RingLoop {
  static constexpr int XB = BM * 128, WB = BN * 128;
  static constexpr int XS = 3 * (XB + WB) <= 160 << 10 ? 3 : 2;
  static constexpr int W_AT = XS * XB, BYTES = W_AT + 3 * WB;
  static constexpr int B = FP8 ? 32 : 16, UNITS = FP8 ? 2 : 1;
  static constexpr int READS = MB + NB;
  // loads that may be on their way while a chunk is read
  static constexpr int AHEAD = XS == 2 ? LW : LX + LW;
  static_assert(BYTES <= 160 << 10, "LDS");

  using Acc = __attribute__((ext_vector_type(B * B / 64))) float;
  struct Frag {
    short8_t x[MB][UNITS], w[NB][UNITS];
  };
  Acc acc[NB][MB];
  int x_at, w_at;

  // read i of a step
  DEV void read(Frag& f, const char* x, const char* w, int step, int i) {
    #pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      const int k = FP8 ? (step * 2 + u) << 5 : step << 6;
      if (i < MB)
        f.x[i][u] = *reinterpret_cast<const short8_t*>(x + (x_at ^ k) +
                                                       i * B * 128);
      else
        f.w[i - MB][u] = *reinterpret_cast<const short8_t*>(
            w + (w_at ^ k) + (i - MB) * B * 128);
    }
  }
  DEV void product(const Frag& f, int n, int m) {
    if constexpr (FP8) {
      union { short8_t s[2]; int32x8_t v; } u{{f.w[n][0], f.w[n][1]}},
          v{{f.x[m][0], f.x[m][1]}};
      acc[n][m] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
          u.v, v.v, acc[n][m], 0, 0, 0, 0, 0, 0);    // e4m3, no scales
    } else {
      acc[n][m] = mfma16(f.w[n][0], f.x[m][0], acc[n][m]);
    }
  }

  // The products of rows x_row and w_row of the tile on.  x_load(l, d, i) and
  // w_load(l, d, i) issue load i of chunk d to the slot l.  Every wave has to call
  // this; those that are not live only load.
  template <class X, class W>
  DEV void run(char* lds, int x_row, int w_row, int chunks, bool live,
               X x_load, W w_load) {
    const int lane = threadIdx.x & 63;
    x_at = chunk_unit(x_row + lane % B, lane / B);
    w_at = chunk_unit(w_row + lane % B, lane / B);
    #pragma unroll
    for (int n = 0; n < NB; ++n)
      #pragma unroll
      for (int m = 0; m < MB; ++m) acc[n][m] = Acc(0.f);
    #pragma unroll
    for (int i = 0; i < LX; ++i) x_load(lds, 0, i);
    #pragma unroll
    for (int i = 0; i < LW; ++i) w_load(lds + W_AT, 0, i);
    if (chunks > 1) {
      if constexpr (XS > 2)
        #pragma unroll
        for (int i = 0; i < LX; ++i) x_load(lds + XB, 1, i);
      #pragma unroll
      for (int i = 0; i < LW; ++i) w_load(lds + W_AT + WB, 1, i);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(AHEAD) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    }
    // slots of this chunk, and of the one before, which are free
    int xs = 0, ws = 0, x_free = XS - 1, w_free = 2;
    // The loads of chunk d between the products of a step: those of x after the barrier
    // that chunk d begins with, for their time is shorter, then those of w.
    constexpr int Q = NB * MB;
    auto loads = [&](int d, bool after, int q) {
      if (after) {
        #pragma unroll
        for (int i = 0; i < LX; ++i)
          if (i * Q / LX == q && d + XS - 1 < chunks)
            x_load(lds + x_free * XB, d + XS - 1, i);
      } else {
        #pragma unroll
        for (int i = 0; i < LW; ++i)
          if (i * Q / LW == q && d + 2 < chunks)
            w_load(lds + W_AT + w_free * WB, d + 2, i);
      }
    };
    Frag f[2];
    // the products of f, and between them the reads of the step after it, g, and loads
    auto step = [&](const Frag& f, Frag& g, const char* x, const char* w, int k,
                    bool more, int d, bool after) {
      #pragma unroll
      for (int q = 0; q < Q; ++q) {
        if (live) product(f, q / MB, q % MB);
        if (live && more) {
          #pragma unroll
          for (int i = 0; i < READS; ++i)
            if (i * (Q * 3 / 4) / READS == q) read(g, x, w, k, i);
        }
        loads(d, after, q);
        if (live) __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (live) {
      #pragma unroll
      for (int i = 0; i < READS; ++i) read(f[0], lds, lds + W_AT, 0, i);
    }
    #pragma unroll
    for (int i = 0; i < LX; ++i)
      if (XS - 1 < chunks) x_load(lds + x_free * XB, XS - 1, i);
    for (int d = 0; d < chunks; ++d) {
      step(f[0], f[1], lds + xs * XB, lds + W_AT + ws * WB, 1, true, d, false);
      x_free = xs;
      w_free = ws;
      xs = xs == XS - 1 ? 0 : xs + 1;
      ws = ws == 2 ? 0 : ws + 1;
      // chunk d + 1 has landed and all of d has been read, by every wave: its slots
      // are free
      if (d + 2 < chunks)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                     ::"n"(AHEAD) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier"
                     ::: "memory");
      step(f[1], f[0], lds + xs * XB, lds + W_AT + ws * WB, 0, d + 1 < chunks,
           d + 1, true);
    }
    // as above
    in_order();
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
    in_order();
  }
  DEV void in_order() {
    #pragma unroll
    for (int n = 0; n < NB; ++n)
      #pragma unroll
      for (int m = 0; m < MB; ++m) asm volatile("" : "+v"(acc[n][m]));
  }
};

// The sums of 16 x 16 products: a lane has 4 consecutive rows of w of every block of
// 16, (lane >> 4) * 4 on, and row lane & 15 of x.  Rows of w lie in LDS such that those
// of two blocks are 8 outputs beside each other, so that a store has 16 bytes a lane
// and 64 of a row: 256 x 256 tiles of 8192 rows of 28672 x 4096 with 8 bytes a lane, 32
// of a row, 10 us a tile for the stores alone, so 3.
//
// Row of w of row r in LDS: of 32 outputs, and of 32 gates and their 32 up rows, `up`
// rows on.
DEV int plain_row(int r) {
  return (r & ~31) | (r >> 2 & 3) << 3 | (r >> 4 & 1) << 2 | (r & 3);
}
DEV int gated_row(int r, int up) {
  return (r >> 6) * 32 + ((r >> 2 & 3) << 3 | (r >> 5 & 1) << 2 | (r & 3)) +
         (r & 16 ? up : 0);
}
// this lane's outputs of its row of block m of x, whose first output is at `out`, of
// `left` that there are
template <bool GATED, int NB, int MB>
DEV void store_row(const f32x4_t (&acc)[NB][MB], int m, bf16* out, int left) {
  const int at = (threadIdx.x & 63) >> 4 << 3;
  constexpr int EACH = GATED ? 2 : 1;          // blocks of 4 outputs a lane
  #pragma unroll
  for (int n = 0; n < NB; n += 2 * EACH) {
    unsigned v[4];
    #pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4_t y = acc[n + h * EACH][m];
      if constexpr (GATED) {
        #pragma unroll
        for (int j = 0; j < 4; ++j)
          y[j] = y[j] / (1.f + __expf(-y[j])) * acc[n + 2 * h + 1][m][j];
      }
      v[2 * h] = cvt_pk_bf16(y[0], y[1]);
      v[2 * h + 1] = cvt_pk_bf16(y[2], y[3]);
    }
    if (n * (16 / EACH) + at < left)
      *reinterpret_cast<uint4*>(out + n * (16 / EACH) + at) =
          uint4{v[0], v[1], v[2], v[3]};
  }
}
// the same of a part, floats
template <int NB, int MB>
DEV void store_part(const f32x4_t (&acc)[NB][MB], int m, float* out, int left) {
  const int at = (threadIdx.x & 63) >> 4 << 3;
  #pragma unroll
  for (int n = 0; n < NB; n += 2)
    if (n * 16 + at < left) {
      *reinterpret_cast<f32x4_t*>(out + n * 16 + at) = acc[n][m];
      *reinterpret_cast<f32x4_t*>(out + n * 16 + at + 4) = acc[n + 1][m];
    }
}

// The same for 32 x 32 products with scales: a lane has 4 of every 8 rows of w, and two
// such are 8 outputs beside each other.
DEV int plain_row_32(int r) {
  return (r & ~15) | (r >> 2 & 1) << 3 | (r >> 3 & 1) << 2 | (r & 3);
}
template <int NB, int MB>
DEV void store_row_32(const f32x16_t (&acc)[NB][MB], int m, bf16* out,
                      float x_scale, const float* w_scale) {
  const int at = (threadIdx.x & 63) >> 5 << 3;
  #pragma unroll
  for (int n = 0; n < NB; ++n)
    #pragma unroll
    for (int r = 0; r < 16; r += 8) {
      const int c = n * 32 + r * 2 + at;
      float y[8];
      load_vec<float, 8>(w_scale + c, y);
      #pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = acc[n][m][r + j] * x_scale * y[j];
      *reinterpret_cast<uint4*>(out + c) =
          uint4{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3]),
                cvt_pk_bf16(y[4], y[5]), cvt_pk_bf16(y[6], y[7])};
    }
}
