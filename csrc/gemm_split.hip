// out[M, N] = x[M, K] w[N, K]^T for tens to hundreds of rows (gfx950), bf16 in
// and out, float sums; or e4m3 in, with scales of the rows, for up to 128 rows.
//
// A product of 256 rows with 4096 outputs is 64 tiles of 128 x 128, a quarter
// of the compute units; so K is divided too, until there is about one workgroup
// a unit, and a second kernel adds the parts, floats.  Chunks of x and w, 128
// or 256 bytes of a row, go from memory to LDS directly, 16 bytes a lane, into
// a ring that fills most of LDS.
//
// What bounds it: w from memory up to about 100 rows (5.5 TB/s in parts, 5.9 in
// one wave of tiles, as 28672 x 4096, and 4.8 of e4m3), then what the tiles take
// from L2, so that 128 x 128 beat 128 x 64 where K is long, and the
// narrow ones, with longer chunks, where it is short; then the products.  A
// ring of 5 stages, or of chunks twice as long, takes as long, and waves that divide
// a stage's chunks up to 5 % longer.
//
// us, library and here, x and w from memory; more than 256 rows with an activation or
// in parts, and from 129 on with long columns, are csrc/gemm_wide.hip's where its rules
// take them (4096 x 14336 256 rows 45, 512 66):
//   4096 x 14336  32 rows 33 26, 96 68 38, 192 112 46, 256 66 52, 512 98 70
//   6144 x 4096   96 rows 24 23, 192 35 28, 256 44 29
//   4096 x 4096   32 rows 14 11, 96 23 16, 192 34 21, 256 23 23
//   2048 x 7168   32 rows 19 11, 96 20 15, 192 26 19, 256 26 22, 512 33 32
//   5120 x 8192   32 rows 27 22, 96 39 28, 192 64 36, 256 79 38
// silu(gate) * up of the halves, product and activation and here: 28672 x 4096 1 row
//   64 41, 17 rows 52 41, 64 53 42, 128 61 53; 14336 x 2048 32 rows 18 13, 256 33 24;
//   in tiles of 256 x 128 28672 x 4096 256 rows 80 69, 14336 x 1664 512 37 30
// e4m3, with the norm that adds up the parts: 4096 x 14336 16 rows 27 19, 64 31
// 21, 128 44 28; 4096 x 4096 16 rows 15 12, 128 18 15; without: 28672 x 4096 16
// rows 34 23, 64 31 24 (27 in tiles of 64 x 64, of which 448 are not one wave);
// 14336 x 2048 64 rows 14 10; 64 of 6144 x 4096 13.4 11.3, 3072 x 2048 10.7 7.2.
#include "tile_loop.h"

namespace {

struct Split {
  bf16* out;
  float* part;                 // [splits, M, N] with splits > 1
  const void* x;
  const void* w;
  const float* x_scale;        // FP8: of a row of x, and of a row of w
  const float* w_scale;
  int M, N, K;
  long xs, ws;                 // row strides
  int mt, nt, splits;          // tiles of rows, of outputs, parts of K
  bool apart;                  // workgroups of a part begin at columns of their own
};

// BM rows of x, BN of w; WM * WN waves have BM / WM by BN / WN.  A stage has
// KC chunks of 64 columns.  Two waves a SIMD (128 threads are less) keep the
// sums in vector registers.  AUX: of the loads of w.
template <int BM, int BN, int WM, int WN, int STAGES, int KC, bool FP8,
          bool GATED, int AUX>
__global__ __launch_bounds__(WM * WN * 64, 2)
void gemm_split_kernel(Split a) {
  using Loop = TileLoop<BM, BN, WM, WN, STAGES, KC, FP8>;
  constexpr int ELEM = FP8 ? 1 : 2;
  constexpr int LX = Loop::LX, LW = Loop::LW, NI = Loop::NI, MI = Loop::MI;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  // workgroups go to the 8 XCDs in turn: those of one tile of w, which differ
  // in the rows of x, to the same, whose L2 then has it
  const int at = blockIdx.x >> 3;
  const int u = at / a.mt * 8 + (blockIdx.x & 7);
  if (u >= a.nt * a.splits) return;
  constexpr int OUT = GATED ? BN / 2 : BN;                 // outputs
  const int m0 = at % a.mt * BM, n0 = u / a.splits * OUT, z = u % a.splits;
  const int outs = GATED ? a.N >> 1 : a.N;
  const int all = a.K * ELEM / (128 * KC);
  const int first = (int)((long)all * z / a.splits);
  const int chunks = (int)((long)all * (z + 1) / a.splits) - first;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hf = lane >> 5;
  const int wm = wid / WN, wn = wid % WN;
  const bool live = m0 + wm * (BM / WM) < a.M;

  // this lane's 16 bytes of row lane / 8 of each 1-KB load; rows past the end
  // are the last one
  const RowLoads x_rows(static_cast<const char*>(a.x) + m0 * a.xs * ELEM +
                        first * (128 * KC));
  const RowLoads w_rows(static_cast<const char*>(a.w) + n0 * a.ws * ELEM +
                        first * (128 * KC));
  unsigned x_off[LX], w_off[LW];
  #pragma unroll
  for (int j = 0; j < LX; ++j) {
    const int r = (wid * LX + j) * 8 + (lane >> 3);
    x_off[j] = (unsigned)(min(r, a.M - 1 - m0) * a.xs * ELEM) +
               ((lane & 7) ^ (r >> 1 & 7)) * 16;
  }
  #pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int r = (wid * LW + j) * 8 + (lane >> 3);
    // gated: 8 gate rows, then their 8 up rows
    const int n = min(GATED ? (r >> 4) * 8 + (r & 7) : r, outs - 1 - n0) +
                  (GATED && r & 8 ? outs : 0);
    w_off[j] = (unsigned)(n * a.ws * ELEM) + ((lane & 7) ^ (r >> 1 & 7)) * 16;
  }
  // workgroups begin at different columns, so that not all of them ask the same
  // channels of memory at once: 64 rows of 28672 x 4096 46 -> 42 us; those of parts of
  // K only where that matters (few_channels, below).  Those of one tile of w begin at
  // the same, which costs up to 3 % in places (192 rows of 14336 x 2048 gated 23.1 ->
  // 23.7, 96 of 28672 x 4096 49.2 49.0), so that a row's sums do not depend on its place
  // among the rows.  Not those that wait for x: 256 decoded tokens, where 6144 x 4096
  // takes this kernel, 3245 us, with it 3251; 512 rows of 5120 x 8192 in 3 parts of 256 x
  // 128 tiles 49 67
  const int turn = !(BM == 64 || GATED) ? 0
      : a.splits == 1 ? at / a.mt * a.mt % chunks
      : a.apart ? u / a.splits % chunks : 0;
  // load i of a stage: first those of x, then those of w
  auto stage = [&](int slot, int d, int i) {
    d += turn;
    if (d >= chunks) d -= chunks;
    const int s = i % KC;
    char* base = lds + slot * Loop::STAGE + s * Loop::SUB;
    if (i < LX * KC) {
      const int j = i / KC;
      x_rows.to_lds(base + (wid * LX + j) * 1024, x_off[j],
                    (d * KC + s) * 128);
    } else {
      const int j = i / KC - LX;
      w_rows.to_lds<AUX>(base + BM * 128 + (wid * LW + j) * 1024, w_off[j],
                         (d * KC + s) * 128);
    }
  };
  Loop loop;
  loop.run(lds, wm, wn, chunks, live, stage);
  auto& acc = loop.acc;

  // acc[n][m][r]: row (r >> 2) * 8 + hf * 4 + (r & 3) of w of block n, row col
  // of x of block m
  #pragma unroll
  for (int m = 0; m < MI; ++m) {
    const int row = m0 + (wm * MI + m) * 32 + col;
    if (row >= a.M) continue;
    const float xs = FP8 ? a.x_scale[row] : 1.f;
    #pragma unroll
    for (int n = 0; n < NI; ++n) {
      if constexpr (GATED) {
        #pragma unroll
        for (int r = 0; r < 16; r += 8) {
          const int c = n0 + (wn * NI + n) * 16 + r + hf * 4;
          if (c >= outs) continue;
          float y[4];
          #pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float g = acc[n][m][r + j], u = acc[n][m][r + 4 + j];
            y[j] = g / (1.f + __expf(-g)) * u;
          }
          *reinterpret_cast<uint2*>(a.out + (long)row * outs + c) =
              uint2{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3])};
        }
        continue;
      }
      #pragma unroll
      for (int r = 0; r < 16; r += 4) {
        const int c = n0 + (wn * NI + n) * 32 + r * 2 + hf * 4;
        if (c >= a.N) continue;                  // N is a multiple of 4
        f32x4_t y{acc[n][m][r], acc[n][m][r + 1], acc[n][m][r + 2],
                  acc[n][m][r + 3]};
        if constexpr (FP8) {
          const f32x4_t ws = *reinterpret_cast<const f32x4_t*>(a.w_scale + c);
          #pragma unroll
          for (int i = 0; i < 4; ++i) y[i] = y[i] * xs * ws[i];
        }
        if (a.splits > 1)
          *reinterpret_cast<f32x4_t*>(
              a.part + ((long)z * a.M + row) * a.N + c) = y;
        else
          *reinterpret_cast<uint2*>(a.out + (long)row * a.N + c) =
              uint2{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3])};
      }
    }
  }
}

// the parts' sum, 4 outputs a thread
template <int SPLITS>
__global__ __launch_bounds__(256) void gemm_sum_kernel(
    bf16* __restrict__ out, const float* __restrict__ part, long quads) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= quads) return;
  f32x4_t x[SPLITS];
  #pragma unroll
  for (int z = 0; z < SPLITS; ++z)
    x[z] = reinterpret_cast<const f32x4_t*>(part)[z * quads + i];
  #pragma unroll
  for (int z = 1; z < SPLITS; ++z) x[0] += x[z];
  reinterpret_cast<uint2*>(out)[i] =
      uint2{cvt_pk_bf16(x[0][0], x[0][1]), cvt_pk_bf16(x[0][2], x[0][3])};
}

// Whether the workgroups of a product in parts, if they begin together, ask few
// channels of memory: 256 bytes are one channel's, and 32 KB go through all 128.  Rows a
// multiple of 4 KB apart begin on 8 channels or fewer, and every part on others, unless
// they begin a multiple of 4 KB apart too.  1 and 32 rows of w in tiles of 64 x 64, 500
// sizes in 2 to 8 parts, K of 4096 to 28672, time with columns of their own over that
// without: 2 to 4 channels 0.78 (8192 x 16384 70 -> 46 us, 4096 x 14336 in rows of 32 KB
// 38.7 -> 21.9, 5120 x 16384 37 -> 30), 6 0.95 (5120 x 8192 18.2 16.7), 8 0.86 (8192 x
// 28672 90 -> 70, 8192 x 12288 43 -> 34, 5120 x 6144 14.9 12.9, e4m3 5120 x 12288 16.2
// 14.3), 12 of rows of 16 KB 0.9 (2560 x 8192), of others 1.0, 16 and more 1.0 (4096 x
// 14336 21.3 21.7).  Where rows lie no multiple of 4 KB apart the mean of 270 is 1.0 too,
// and single sizes are 10 % faster or slower (8192 x 22016 72 -> 66, 8192 x 16128 1.13).
bool few_channels(long row_bytes, long stretches, int splits) {
  const long period = row_bytes % 32768 ? row_bytes & -row_bytes : 32768;
  if (period < 4096 || period >= 16384) return period >= 16384;
  unsigned begins = 0;         // of the stretches of a period
  for (long z = 0; z < splits; ++z)
    begins |= 1u << stretches * z / splits % (period / 256);
  return 32768 / period * __builtin_popcount(begins) <= 8;
}

}  // namespace

// Tiles of bm rows of x by bn of w: 64 x 64, 64 x 128, 128 x 64, 128 x 128, 256 x
// 128; with scales x and w are e4m3, in tiles of 64 x 32, 64 x 64 or 64 x 128.
// out contiguous; rows of K of 256 bytes, N a multiple of 4; rows of x and w 16-byte
// aligned; splits 1 to 8, at most one a 256 bytes, part with more than one.
// Without out the parts are left for the norm that adds them up.  gated, of
// bfloat16 without parts: out = silu(gate) * up of the halves of w, whose rows
// are a multiple of 8.
void launch_gemm_split(bf16* out, float* part, const void* x, const void* w,
                       const float* x_scale, const float* w_scale, int M,
                       int N, int K, long xs, long ws, int bm, int bn,
                       int splits, bool gated, hipStream_t stream) {
  // A tile of w that several tiles of rows share is read once where they go through
  // it together.  One that has few rows does not keep step, for the rows past the end
  // cost it nothing, and non-temporal loads leave the others nothing.  us, plain and
  // so: 128 rows a tile, 129 rows of 4096 x 14336 43 49, 192 43 47, 256 46.5 45, 257
  // 69 80, 350 74 73, 420 71 81,
  // 480 77.5 77; 256 a tile, 320 55.6 55.8, 512 62.5 59.5.
  const int last = (M - 1) % bm + 1;
  const bool once = M <= bm || last * 4 >= bm * 3;
  const int size = x_scale ? 1 : 2;
  Split a{out, part, x, w, x_scale, w_scale, M, N, K, xs, ws, 0, 0, splits,
          few_channels(ws * size, (long)K * size / 256, splits)};
  #define WITH(BM, BN, WM, WN, STAGES, KC, FP8, GATED, AUX)                 \
    {                                                                       \
      constexpr int BYTES = STAGES * KC * (BM + BN) * 128;                  \
      constexpr auto kernel =                                               \
          &gemm_split_kernel<BM, BN, WM, WN, STAGES, KC, FP8, GATED, AUX>;  \
      static const hipError_t set = hipFuncSetAttribute(                    \
          reinterpret_cast<const void*>(kernel),                            \
          hipFuncAttributeMaxDynamicSharedMemorySize, BYTES);               \
      HIP_CHECK(set);                                                       \
      a.mt = (M + BM - 1) / BM;                                             \
      a.nt = (N + BN - 1) / BN;                                             \
      const unsigned units = (unsigned)(a.nt * splits + 7) / 8 * 8;         \
      kernel<<<units * a.mt, WM * WN * 64, BYTES, stream>>>(a);             \
    }
  #define RUN(BM, BN, WM, WN, STAGES, KC, FP8, GATED)                       \
    {                                                                       \
      if (once) WITH(BM, BN, WM, WN, STAGES, KC, FP8, GATED, ONCE)          \
      else WITH(BM, BN, WM, WN, STAGES, KC, FP8, GATED, 0)                  \
    }
  #define KINDS(BM, BN, WM, WN, STAGES, KC)                                 \
    {                                                                       \
      if (gated) RUN(BM, BN, WM, WN, STAGES, KC, false, true)               \
      else RUN(BM, BN, WM, WN, STAGES, KC, false, false)                    \
    }
  if (x_scale) {
    // two workgroups a unit, with half the ring each, where there are as many
    if (bn == 32)
      RUN(64, 32, 2, 1, 3, 2, true, false)
    else if (bn == 128)
      RUN(64, 128, 2, 2, 3, 2, true, false)
    else if ((long)((M + 63) / 64) * ((N + 63) / 64) * splits > 256)
      RUN(64, 64, 2, 2, 2, 2, true, false)
    else
      RUN(64, 64, 2, 2, 4, 2, true, false)
  } else if (bm == 256)
    KINDS(256, 128, 4, 2, 3, 1)
  else if (bm == 128 && bn == 128)
    KINDS(128, 128, 2, 4, 4, 1)
  else if (bm == 128)
    KINDS(128, 64, 4, 2, 3, 2)
  else if (bn == 128)
    KINDS(64, 128, 2, 2, 3, 2)
  else
    KINDS(64, 64, 2, 2, 4, 2)
  #undef KINDS
  #undef RUN
  #undef WITH
  if (splits == 1 || !out) return;
  const long quads = (long)M * N / 4;
  #define SUM(S)                                                            \
    case S:                                                                 \
      gemm_sum_kernel<S><<<(unsigned)((quads + 255) / 256), 256, 0,         \
                           stream>>>(out, part, quads);                     \
      break;
  switch (splits) {
    SUM(2) SUM(3) SUM(4) SUM(5) SUM(6) SUM(7) SUM(8)
    default: throw std::runtime_error("gemm_split: 1 to 8 parts");
  }
  #undef SUM
}
