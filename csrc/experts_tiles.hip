// Grouped expert products in LDS tiles (gfx950), bf16 or e4m3 with scales.
//
//   out[p, n] = x[r] . w[e, n] of every choice, in the order of experts.hip's
//   sort with bm rows a tile: r is p, or with div the token order[p] / div
//   GATED: out[p, i] = silu(x[r] . w[e, i]) * (x[r] . w[e, N + i])
//
// A workgroup has bm choices of one expert and BN rows of its weights, K in
// chunks of 128 bytes.  Both go from memory to LDS directly, 16 bytes a lane
// and whole 128-byte lines, into a ring of chunks; weights are the A operand of
// matrix products, so that a lane's results are consecutive outputs of one choice,
// and rows of gates and their up rows alternate in LDS: both of a pair are in one
// lane, and the activation needs no pass of its own.  Tiles of 64 and 128 choices
// form 32 x 32 products, with 8 gates and their 8 up rows in turn; those of up to 256
// (experts_high_kernel) 16 x 16 of bf16, with 16 and 16.
//
// What bounds it: the weights' bytes up to about 100 choices an expert, so bm
// is what covers most counts, then the products.  Mixtral 8x7B layer (8 experts,
// 14336 x 4096, 2.8 GB), us: 16 choices an expert 443, 48 470, 112 566, 140 601, 302
// 906, 500 1210.  32 experts of 1024 x 2048, 64 choices 93.
#include <algorithm>
#include <type_traits>

#include "tile_loop.h"

namespace {

struct Tiles {
  bf16* out;
  const void* x;
  const void* w;
  const float* x_scale;        // FP8: of a row of x, and of a row of w
  const float* w_scale;
  const int* order;
  const int* expert;
  int N, K, div, nx;           // N outputs a choice, nx blocks of them
};

DEV int row_of(const Tiles& a, int p) {
  const int choice = a.order[p];
  return a.div ? (choice >= 0 ? choice / a.div : 0) : p;
}

// The sums of a wave, of choices p0 on and outputs n0 on.  acc[n][m][r]: weight row
// (r >> 2) * 8 + hf * 4 + (r & 3) of block n, choice col of block m.
template <bool GATED, bool FP8, int NI, int MI>
DEV void store_tile(const Tiles& a, const f32x16_t (&acc)[NI][MI], int e,
                    int p0, int n0) {
  const int lane = threadIdx.x & 63, col = lane & 31, hf = lane >> 5;
  #pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int p = p0 + m * 32 + col;
    if (a.order[p] < 0) continue;
    bf16* op = a.out + (long)p * a.N + n0 + hf * 4;
    const float xs = FP8 ? a.x_scale[row_of(a, p)] : 1.f;
    #pragma unroll
    for (int n = 0; n < NI; ++n) {
      if constexpr (GATED) {
        #pragma unroll
        for (int r = 0; r < 16; r += 8) {
          float y[4];
          #pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float g = acc[n][m][r + j], u = acc[n][m][r + 4 + j];
            y[j] = g / (1.f + __expf(-g)) * u;
          }
          *reinterpret_cast<uint2*>(op + n * 16 + r) =
              uint2{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3])};
        }
      } else {
        #pragma unroll
        for (int r = 0; r < 16; r += 4) {
          float y[4];
          #pragma unroll
          for (int j = 0; j < 4; ++j) y[j] = acc[n][m][r + j];
          if constexpr (FP8) {
            const float4 ws = *reinterpret_cast<const float4*>(
                a.w_scale + (long)e * a.N + n0 + n * 32 + r * 2 + hf * 4);
            y[0] = y[0] * xs * ws.x;
            y[1] = y[1] * xs * ws.y;
            y[2] = y[2] * xs * ws.z;
            y[3] = y[3] * xs * ws.w;
          }
          *reinterpret_cast<uint2*>(op + n * 32 + r * 2) =
              uint2{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3])};
        }
      }
    }
  }
}

constexpr int HIGH_BYTES = 160 << 10;      // of LDS

// BM choices, BN rows of weights; WM * WN waves have BM / WM by BN / WN
template <int BM, int BN, int WM, int WN, int STAGES, bool GATED, bool FP8,
          bool FAR>
__global__ __launch_bounds__(WM * WN * 64,
                             WM * WN == 4 ? 2 : WM * WN / 4)
void experts_tiles_kernel(Tiles a) {
  using Loop = TileLoop<BM, BN, WM, WN, STAGES, 1, FP8>;
  constexpr int LX = Loop::LX, LW = Loop::LW;
  constexpr int OUT = GATED ? BN / 2 : BN;                 // outputs
  constexpr int ELEM = FP8 ? 1 : 2;
  static_assert(!(GATED && FP8), "the activation's scale needs whole rows");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tile = blockIdx.x / a.nx, nb = blockIdx.x % a.nx;
  const int tiles = gridDim.x / a.nx;
  const int e = a.expert[tile];
  const int last = a.expert[max(tile - 1, 0)];
  const int next = a.expert[min(tile + 1, tiles - 1)];
  if (e < 0) return;
  // Weights that one tile takes are read once (ONCE), those of several not: they
  // would leave the others nothing.  us, up and down, in tiles of 128, of 8 experts of
  // 14336 x 4096, 112 choices each 718 -> 660, of 16 of 2048 x 4096 226 -> 214.  Where
  // tokens prefer the same experts, tiles are several, by ONCE and so: 300 choices of
  // each of 2 experts of 16 in tiles of 64 95 -> 71, 64 experts of 1024 x 2048, up to
  // 190 each 104 -> 92, 150 of each of 2 of 8 343 -> 305, 100 to 200 uneven tokens of
  // 8 604 -> 577 and 606 -> 588; even ones 440 442, 138 138, 149 149.
  const bool alone = ((tile == 0) | (last != e)) &
                     ((tile + 1 == tiles) | (next != e));
  const int n0 = nb * OUT, p0 = tile * BM;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // a SIMD has waves of different choices: those without any do nothing
  const int wm = wid / WN, wn = wid % WN;
  const bool live = a.order[p0 + wm * (BM / WM)] >= 0;

  // this lane's 16 bytes of row lane / 8 of each 1-KB load
  const int lr = lane >> 3;
  auto column = [&](int r) { return ((lane & 7) ^ (r >> 1 & 7)) * 16; };
  const long row_bytes = (long)a.K * ELEM;
  auto w_row = [&](int r) {    // gated: 8 gate rows, then their 8 up rows
    return GATED ? (r >> 4) * 8 + (r & 7) + (r & 8 ? a.N : 0) : r;
  };
  const char* w0 = static_cast<const char*>(a.w) +
                   ((long)e * (GATED ? 2 * a.N : a.N) + n0) * row_bytes;
  const char* x0 = static_cast<const char*>(a.x) + (a.div ? 0 : p0 * row_bytes);
  const RowLoads x_rows(x0), w_rows(w0);
  long x_off[LX], w_off[LW];   // below 4 GB but for FAR
  #pragma unroll
  for (int j = 0; j < LX; ++j) {
    const int r = (wid * LX + j) * 8 + lr;
    x_off[j] = (row_of(a, p0 + r) - (a.div ? 0 : p0)) * row_bytes + column(r);
  }
  #pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int r = (wid * LW + j) * 8 + lr;
    w_off[j] = w_row(r) * row_bytes + column(r);
  }
  auto load = [&](auto once, char* l, const RowLoads& rows, const char* base,
                  long off, int d) {
    constexpr int AUX = decltype(once)::value ? ONCE : 0;
    if constexpr (FAR)
      __builtin_amdgcn_global_load_lds(
          (__attribute__((address_space(1))) const unsigned*)(base + off +
                                                              d * 128),
          (__attribute__((address_space(3))) unsigned*)l, 16, 0, AUX);
    else
      rows.to_lds<AUX>(l, (unsigned)off, d * 128);
  };
  // Where the weights are the bound workgroups begin at different columns, so
  // that not all of them ask the same channels of memory at once; those of one
  // expert and the same outputs at the same.  192 tokens of 2 choices, 8 experts
  // of 14336 x 4096 355 + 188 -> 321 + 162 us; 4 of 32 of 1024 x 2048 65 + 29 ->
  // 50 + 29.
  // Three times as far apart where rows are long: 140 random sizes (4 to 64
  // experts, K of 1024 to 14336), time over that of once as far: rows of 12 KB and
  // more 0.984, 8 and 10 KB in tiles of 128 0.985, of 64 1.02 (16 of 4096 x 4096,
  // 22 choices each, 99 108), shorter ones 1.01 (64 of 3072 x 2048 150 162).
  const int stages = (int)(row_bytes / 128);
  const int apart = stages >= (BM == 64 ? 96 : 64) ? 3 : 1;
  const int turn = (nb + e * a.nx) / 8 * apart % stages;
  // load i of a stage: first those of x, then those of w
  auto stage = [&](auto once, int slot, int d, int i) {
    d += turn;
    if (d >= stages) d -= stages;
    char* l = lds + slot * Loop::STAGE;
    if (i < LX)
      load(std::false_type(), l + (wid * LX + i) * 1024, x_rows, x0, x_off[i],
           d);
    else
      load(once, l + BM * 128 + (wid * LW + i - LX) * 1024, w_rows, w0,
           w_off[i - LX], d);
  };
  Loop loop;
  auto run = [&](auto once) {
    loop.run(lds, wm, wn, stages, live, [&](int slot, int d, int i) {
      stage(once, slot, d, i);
    });
  };
  if (alone)
    run(std::true_type());
  else
    run(std::false_type());
  store_tile<GATED, FP8>(a, loop.acc, e, p0 + wm * (BM / WM),
                         n0 + wn * (OUT / WN));
}

// A tile of up to 256 choices, as high as it has choices: H blocks of 32, and BN rows
// of weights.  Of the 8 waves 4 have the first blocks of every kind, 4 the others, MB
// each, and the two of a SIMD are one of both, so that all SIMDs have the same
// products if H is odd too.  bf16: 2 of the 4 share the choices, and every second wave
// has the same half of the weights; blocks of 16.  e4m3: each has a quarter of the
// weights; blocks of 32.  What is not there is neither formed nor loaded.
//
// What bounds it: 160 x 256 what a unit loads, 52 KB a chunk at some 45 GB/s, and the
// products (8 experts of 14336 x 4096, 302 choices each, up 500 us without products, 440
// without loads, 613 with both), larger ones power.  us, with tiles of 256 of which the
// last of an expert is mostly padding, two stages and 32 x 32 products, and here, up and
// down: 302 choices 743 431 and 613 293, 512 872 473 and 817 394, 2000 3168 1593 and
// 2912 1428, 130 454 232 and 430 211; 16 of 2048 x 4096, 300 239 132 and 170 95; 32 of
// 1024 x 2048, 300 131 89 and 92 67, 1000 264 169 and 255 147.  e4m3: 302 404 216 and
// 335 146, 2000 1815 943 and 1671 752.  Even: two workgroups of one expert with its
// choices together and half of the weights each.
template <int H, bool LATER, int BN, bool GATED, bool FP8, bool FAR>
DEV void high_tile_part(const Tiles& a, char* lds, int e, int p0, int nb,
                        bool alone) {
  constexpr int BM = H * 32, OUT = GATED ? BN / 2 : BN;
  constexpr int MB = LATER ? H / 2 : H - H / 2, FIRST = LATER ? H - H / 2 : 0;
  constexpr int PARTS = FP8 ? 4 : 2;           // of the weights
  constexpr int B = FP8 ? 32 : 16, NB = BN / PARTS / B, LW = BN / 64;
  constexpr int ROWS = MB ? MB : 1;
  using Loop = RingLoop<BM, BN, ROWS, NB, MB, LW, FP8>;
  const int n0 = nb * OUT;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wid % PARTS;
  const int x_row = FIRST * 32 + (wid & 3) / PARTS * (MB * B);
  const int lr = lane >> 3;
  auto column = [&](int r) { return ((lane & 7) ^ (r >> 1 & 7)) * 16; };
  const long row_bytes = (long)a.K * (FP8 ? 1 : 2);
  const char* x0 = static_cast<const char*>(a.x) + (a.div ? 0 : p0 * row_bytes);
  const char* w0 = static_cast<const char*>(a.w) +
                   ((long)e * (GATED ? 2 * a.N : a.N) + n0) * row_bytes;
  const RowLoads x_rows(x0), w_rows(w0);
  using Offset = std::conditional_t<FAR, long, unsigned>;
  Offset x_off[ROWS], w_off[LW];
  #pragma unroll
  for (int j = 0; j < MB; ++j) {
    const int r = FIRST * 32 + ((wid & 3) * MB + j) * 8 + lr;
    x_off[j] = (Offset)((row_of(a, p0 + r) - (a.div ? 0 : p0)) * row_bytes +
                        column(r));
  }
  #pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int r = (wid * LW + j) * 8 + lr;
    const int n = FP8 ? plain_row_32(r) : GATED ? gated_row(r, a.N) : plain_row(r);
    w_off[j] = (Offset)(n * row_bytes + column(r));
  }
  auto load = [&](auto once, char* l, const RowLoads& rows, const char* base,
                  Offset off, int d) {
    constexpr int AUX = decltype(once)::value ? ONCE : 0;
    if constexpr (FAR)
      __builtin_amdgcn_global_load_lds(
          (__attribute__((address_space(1))) const unsigned*)(base + off +
                                                              d * 128),
          (__attribute__((address_space(3))) unsigned*)l, 16, 0, AUX);
    else
      rows.to_lds<AUX>(l, off, d * 128);
  };
  Loop loop;
  const int chunks = (int)(row_bytes / 128);
  auto run = [&](auto once, int turn) {
    // which is 0 at compile time where it is
    const auto at = [&](int d) {
      d += turn;
      return turn && d >= chunks ? d - chunks : d;
    };
    loop.run(lds, x_row, part * (BN / PARTS), chunks, MB > 0,
             [&](char* l, int d, int i) {
               load(std::false_type(), l + (FIRST * 4 + (wid & 3) * MB + i) * 1024,
                    x_rows, x0, x_off[i], at(d));
             },
             [&](char* l, int d, int i) {
               load(once, l + (wid * LW + i) * 1024, w_rows, w0, w_off[i],
                    at(d));
             });
  };
  // Weights of one tile, in rows of 4 KB, and with gates of 8 KB: of one column they are
  // all a few channels'.  So each die, which has every eighth of the tiles of outputs,
  // begins at a column of its own, and its workgroups still share x.  130 to 250 choices
  // an expert, time over that without, two of the same differing by up to 10 %: 4 KB 0.94
  // in 42 sizes (8 experts of 14336 x 2048 up, 150 224 -> 198 us, 16 of 2048 x 2048 73
  // 59, down 16 of 4096 x 2048 76 64, e4m3 8 of 16384 x 4096 148 127), 8 KB with gates
  // 0.94 in 14 (8 of 8192 x 4096, 170 261 220, 8 of 14336 x 4096, 130 396 367) but with
  // few tiles of outputs 1.0; plain ones and e4m3 of 8 KB 1.03, up to 1.2 (16 of 4096 x
  // 4096, 150 138 145, e4m3 8 of 16384 x 8192, 130 246 273).  12 KB 0.95, and with 250
  // choices up to 1.07; 2, 6, 10, 14, 16 KB and more 1.0 to 1.15 (8 of 4096 x 14336, 250
  // 428 454).
  if (!alone)
    run(std::false_type(), 0);
  else if (row_bytes == 4096 ? a.nx >= 8
                             : GATED && row_bytes == 8192 && a.nx >= 16)
    run(std::true_type(), nb % 8 * chunks / 8);
  else
    run(std::true_type(), 0);
  if constexpr (MB > 0 && FP8) {
    #pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int p = p0 + x_row + m * 32 + (lane & 31);
      if (a.order[p] < 0) continue;
      const int c = n0 + part * (OUT / PARTS);
      store_row_32(loop.acc, m, a.out + (long)p * a.N + c,
                   a.x_scale[row_of(a, p)], a.w_scale + (long)e * a.N + c);
    }
  } else if constexpr (MB > 0) {
    #pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int p = p0 + x_row + m * 16 + (lane & 15);
      if (a.order[p] < 0) continue;
      store_row<GATED>(loop.acc, m, a.out + (long)p * a.N + n0 +
                                        part * (OUT / PARTS), OUT / PARTS);
    }
  }
}

template <int BN, bool GATED, bool FP8, bool FAR>
__global__ __launch_bounds__(512, 2) void experts_high_kernel(Tiles a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  int tile = blockIdx.x / a.nx, nb = blockIdx.x % a.nx;
  const int tiles = gridDim.x / a.nx;
  const int e = a.expert[tile];
  const int last = a.expert[max(tile - 1, 0)];
  const int next = a.expert[min(tile + 1, tiles - 1)];
  if (e < 0) return;
  const bool alone = ((tile == 0) | (last != e)) &
                     ((tile + 1 == tiles) | (next != e));
  // The tiles of an expert that take the same weights go to one die together,
  // whose L2 then has them, where an expert has 128 MB of them, half of what the
  // memory's cache holds: later tiles would find them gone.  180 random sizes (2
  // to 16 experts, 100 to 1100 choices each, N of 2048 to 16384, K of 1024 to
  // 15000), time over that without: 256 x 256 from 128 MB on 0.962, two of 29 more
  // than 1.2 % slower (16 of 16384 x 5760, 1060 choices 6666 -> 6335 us, 8 of 16384
  // x 2432, 590 841 -> 767, 8 of 8192 x 14080, 320 1.041), with 50 to 128 MB 0.997,
  // with less 1.024; 256 x 128, which are fewer, 1.032 (2 of 10240 x 3072 77 ->
  // 96).  More than 32 tiles share them without it.
  if (BN == 256 && a.nx % 8 == 0 &&
      (GATED ? 2 : 1) * a.N * ((long)a.K * (FP8 ? 1 : 2)) >= 128l << 20) {
    const int t = threadIdx.x & 63;
    const unsigned long back =
        ~__ballot(t <= tile && a.expert[t <= tile ? tile - t : 0] == e);
    const unsigned long on = ~__ballot(
        tile + t < tiles && a.expert[tile + t < tiles ? tile + t : 0] == e);
    const int before = (back ? __builtin_ctzll(back) : 64) - 1;
    const int count = before + (on ? __builtin_ctzll(on) : 64);
    if (count <= 32) {
      const int at = before * a.nx + nb;
      nb = at / (8 * count) * 8 + at % 8;
      tile += at / 8 % count - before;
    }
  }
  const int p0 = tile * 256;
  const int lane = threadIdx.x & 63;
  // a tile's choices come first, then its padding
  const int high = __builtin_popcountll(
      __ballot(lane < 8 && a.order[p0 + (lane & 7) * 32] >= 0));
  const bool first = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < 4;
  #define HIGH(H)                                                           \
    case H:                                                                 \
      if (first)                                                            \
        high_tile_part<H, false, BN, GATED, FP8, FAR>(a, lds, e, p0, nb,    \
                                                      alone);               \
      else                                                                  \
        high_tile_part<H, true, BN, GATED, FP8, FAR>(a, lds, e, p0, nb,     \
                                                     alone);                \
      break;
  switch (high) {
    HIGH(1) HIGH(2) HIGH(3) HIGH(4) HIGH(5) HIGH(6) HIGH(7) HIGH(8)
  }
  #undef HIGH
}

}  // namespace

// bm 64, 128 or 256; rows of w of 128-byte chunks, at least two; outputs N a
// multiple of 128 (gated: of 64).  x, w and out contiguous; with scales x and
// w are e4m3.
void launch_experts_tiles(bool gated, bf16* out, const void* x, const void* w,
                          const float* x_scale, const float* w_scale,
                          const int* order, const int* expert, int experts,
                          long x_rows, int tiles, int N, int K, int div, int bm,
                          hipStream_t stream) {
  if (tiles == 0) return;
  Tiles a{out, x, w, x_scale, w_scale, order, expert, N, K, div, 0};
  #define RUN(BM, BN, WM, WN, STAGES, GATED, FP8, FAR)                      \
    {                                                                       \
      constexpr int BYTES = STAGES * (BM + BN) * 128;                       \
      static const hipError_t set = hipFuncSetAttribute(                    \
          reinterpret_cast<const void*>(                                    \
              &experts_tiles_kernel<BM, BN, WM, WN, STAGES, GATED, FP8,     \
                                  FAR>),                                   \
          hipFuncAttributeMaxDynamicSharedMemorySize, BYTES);               \
      HIP_CHECK(set);                                                       \
      a.nx = N / (GATED ? BN / 2 : BN);                                     \
      experts_tiles_kernel<BM, BN, WM, WN, STAGES, GATED, FP8, FAR>         \
          <<<(unsigned)(tiles * a.nx), WM * WN * 64, BYTES, stream>>>(a);   \
    }
  #define KINDS(BM, BN, WM, WN, STAGES, FAR)                                \
    {                                                                       \
      if (x_scale) RUN(BM, BN, WM, WN, STAGES, false, true, FAR)            \
      else if (gated) RUN(BM, BN, WM, WN, STAGES, true, false, FAR)         \
      else RUN(BM, BN, WM, WN, STAGES, false, false, FAR)                   \
    }
  #define LAUNCH(BN, GATED, FP8, FAR)                                       \
    {                                                                       \
      constexpr auto kernel = &experts_high_kernel<BN, GATED, FP8, FAR>;    \
      static const hipError_t set = hipFuncSetAttribute(                    \
          reinterpret_cast<const void*>(kernel),                            \
          hipFuncAttributeMaxDynamicSharedMemorySize, HIGH_BYTES);          \
      HIP_CHECK(set);                                                       \
      a.nx = N / (GATED ? BN / 2 : BN);                                     \
      kernel<<<(unsigned)(tiles * a.nx), 512, HIGH_BYTES, stream>>>(a);     \
    }
  #define HIGH(BN, FAR)                                                     \
    {                                                                       \
      if (x_scale) LAUNCH(BN, false, true, FAR)                             \
      else if (gated) LAUNCH(BN, true, false, FAR)                          \
      else LAUNCH(BN, false, false, FAR)                                    \
    }
  // 256 rows of weights need fewer loads of x and LDS reads, 128 make twice the
  // workgroups, a wave of which takes three fifths of the time.  us, 128 and 256, 8
  // experts of 14336 x 4096: down 130 choices each 211 262, 256 255 305 (of 128 tiles
  // of 256), 302 361 293, 512 477 394; up 130 460 430, 302 784 610, 2000 3570 2910; 32
  // of 1024 x 2048 up 300 choices 112 92, 1000 286 255, down 190 47 43, 500 97 75.
  const int wide = gated ? 128 : 256;
  const auto waves = [](long groups) { return (groups + 255) / 256; };
  // tiles with choices, if they are even
  const long all = std::max(experts, 1);
  const long mean = std::max((tiles * 256l - 255 * all) / all, 1l);
  const long live = std::min<long>(tiles, (mean + 255) / 256 * all);
  // what 32 bits of offset do not reach
  const long row_bytes = (long)K * (x_scale ? 1 : 2);
  const bool far = (div ? x_rows : bm) * row_bytes >= 1l << 32 ||
                   (gated ? N + 256l : 256l) * row_bytes >= 1l << 32;
  if (bm == 64) {
    if (far) KINDS(64, 128, 2, 2, 3, true)
    else KINDS(64, 128, 2, 2, 3, false)
  } else if (bm == 128) {
    if (far) KINDS(128, 128, 2, 4, 3, true)
    else KINDS(128, 128, 2, 4, 3, false)
  } else if (far) {
    HIGH(128, true)
  } else if (N % wide == 0 && waves(live * (N / wide)) * 5 <=
                                  waves(live * (N / wide) * 2) * 3) {
    HIGH(256, false)
  } else {
    HIGH(128, false)
  }
  #undef HIGH
  #undef LAUNCH
  #undef KINDS
  #undef RUN
}
