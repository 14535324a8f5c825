// out[M, N] = x[M, K] w[N, K]^T for tens to hundreds of rows (gfx950), bf16 in
// and out, float sums.
//
// A product of 256 rows with 4096 outputs is 64 tiles of 128 x 128, a quarter
// of the compute units; so K is divided too, until there is about one workgroup
// a unit, and a second kernel adds the parts, floats.  Chunks of x and w, 128
// or 256 bytes of a row, go from memory to LDS directly, 16 bytes a lane, into
// a ring that fills most of LDS.
//
// What bounds it: w from memory up to about 100 rows (3.7 TB/s), then what the
// tiles take from L2, so that 128 x 128 beat 128 x 64 where K is long, and the
// narrow ones, with longer chunks, where it is short; then the products.  A
// ring of 5 stages, or of chunks twice as long, takes as long.
//
// us, library and here:
//   4096 x 14336  32 rows 35 27, 96 63 32, 192 102 45, 256 62 49, 512 88 76
//   6144 x 4096   96 rows 23 19, 192 34 28, 256 40 30
//   4096 x 4096   32 rows 13 12, 96 22 14, 192 33 22, 256 23 23
//   2048 x 7168   32 rows 19 11, 96 19 14, 192 25 19, 256 25 20, 512 32 29
//   5120 x 8192   32 rows 25 23, 96 37 26, 192 61 36, 256 72 39
#include "tile_loop.h"

namespace {

struct Split {
  bf16* out;
  float* part;                 // [splits, M, N] with splits > 1
  const bf16* x;
  const bf16* w;
  int M, N, K;
  long xs, ws;                 // row strides
  int mt, nt, splits;          // tiles of rows, of outputs, parts of K
};

// BM rows of x, BN of w; WM * WN waves have BM / WM by BN / WN.  A stage has
// KC chunks of 64 columns.
template <int BM, int BN, int WM, int WN, int STAGES, int KC>
__global__ __launch_bounds__(WM * WN * 64, WM * WN / 4)
void gemm_split_kernel(Split a) {
  using Loop = TileLoop<BM, BN, WM, WN, STAGES, KC, false>;
  constexpr int LX = Loop::LX, LW = Loop::LW, NI = Loop::NI, MI = Loop::MI;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  // workgroups go to the 8 XCDs in turn: those of one tile of w, which differ
  // in the rows of x, to the same, whose L2 then has it
  const int at = blockIdx.x >> 3;
  const int u = at / a.mt * 8 + (blockIdx.x & 7);
  if (u >= a.nt * a.splits) return;
  const int m0 = at % a.mt * BM, n0 = u / a.splits * BN, z = u % a.splits;
  const int all = a.K / (64 * KC);
  const int first = (int)((long)all * z / a.splits);
  const int chunks = (int)((long)all * (z + 1) / a.splits) - first;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hf = lane >> 5;
  const int wm = wid / WN, wn = wid % WN;
  const bool live = m0 + wm * (BM / WM) < a.M;

  // this lane's 16 bytes of row lane / 8 of each 1-KB load; rows past the end
  // are the last one
  const RowLoads x_rows(a.x + m0 * a.xs + first * (64 * KC));
  const RowLoads w_rows(a.w + n0 * a.ws + first * (64 * KC));
  unsigned x_off[LX], w_off[LW];
  #pragma unroll
  for (int j = 0; j < LX; ++j) {
    const int r = (wid * LX + j) * 8 + (lane >> 3);
    x_off[j] = (unsigned)(min(r, a.M - 1 - m0) * a.xs * 2) +
               ((lane & 7) ^ (r >> 1 & 7)) * 16;
  }
  #pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int r = (wid * LW + j) * 8 + (lane >> 3);
    w_off[j] = (unsigned)(min(r, a.N - 1 - n0) * a.ws * 2) +
               ((lane & 7) ^ (r >> 1 & 7)) * 16;
  }
  auto stage = [&](int slot, int d) {
    char* base = lds + slot * Loop::STAGE;
    #pragma unroll
    for (int j = 0; j < LX; ++j)
      #pragma unroll
      for (int s = 0; s < KC; ++s)
        x_rows.to_lds(base + s * Loop::SUB + (wid * LX + j) * 1024, x_off[j],
                      (d * KC + s) * 128);
    #pragma unroll
    for (int j = 0; j < LW; ++j)
      #pragma unroll
      for (int s = 0; s < KC; ++s)
        w_rows.to_lds(base + s * Loop::SUB + BM * 128 + (wid * LW + j) * 1024,
                      w_off[j], (d * KC + s) * 128);
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
    #pragma unroll
    for (int n = 0; n < NI; ++n)
      #pragma unroll
      for (int r = 0; r < 16; r += 4) {
        const int c = n0 + (wn * NI + n) * 32 + r * 2 + hf * 4;
        if (c >= a.N) continue;                  // N is a multiple of 4
        if (a.splits > 1) {
          *reinterpret_cast<f32x4_t*>(
              a.part + ((long)z * a.M + row) * a.N + c) =
              f32x4_t{acc[n][m][r], acc[n][m][r + 1], acc[n][m][r + 2],
                      acc[n][m][r + 3]};
        } else {
          *reinterpret_cast<uint2*>(a.out + (long)row * a.N + c) =
              uint2{cvt_pk_bf16(acc[n][m][r], acc[n][m][r + 1]),
                    cvt_pk_bf16(acc[n][m][r + 2], acc[n][m][r + 3])};
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

}  // namespace

// Tiles of bm rows by bn outputs: 128 x 64, 128 x 128, 256 x 128.  out
// contiguous; K a multiple of 128, N of 4; rows of x and w 16-byte aligned;
// splits 1 to 8, at most K / 128, part with more than one.  Without out the
// parts are left for the norm that adds them up.
void launch_gemm_split(bf16* out, float* part, const bf16* x, const bf16* w,
                       int M, int N, int K, long xs, long ws, int bm,
                       int bn, int splits, hipStream_t stream) {
  Split a{out, part, x, w, M, N, K, xs, ws, 0, 0, splits};
  #define RUN(BM, BN, WM, WN, STAGES, KC)                                   \
    {                                                                       \
      constexpr int BYTES = STAGES * KC * (BM + BN) * 128;                  \
      static const hipError_t set = hipFuncSetAttribute(                    \
          reinterpret_cast<const void*>(                                    \
              &gemm_split_kernel<BM, BN, WM, WN, STAGES, KC>),              \
          hipFuncAttributeMaxDynamicSharedMemorySize, BYTES);               \
      HIP_CHECK(set);                                                       \
      a.mt = (M + BM - 1) / BM;                                             \
      a.nt = (N + BN - 1) / BN;                                             \
      const unsigned units = (unsigned)(a.nt * splits + 7) / 8 * 8;         \
      gemm_split_kernel<BM, BN, WM, WN, STAGES, KC>                           \
          <<<units * a.mt, WM * WN * 64, BYTES, stream>>>(a);               \
    }
  if (bm == 256)
    RUN(256, 128, 4, 2, 3, 1)
  else if (bn == 128)
    RUN(128, 128, 2, 4, 4, 1)
  else
    RUN(128, 64, 4, 2, 3, 2)
  #undef RUN
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
