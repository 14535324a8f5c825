// out[M, N] = x[M, K] w[N, K]^T for hundreds of rows and more (gfx950), bf16, float
// sums; or silu(gate) * up of the halves of w, which saves a pass over both; or float
// parts of K, for the norm that adds them, where tiles alone leave the chip idle.
//
// Even tiles of up to 256 rows by 128 or 256 outputs, whichever wave of them takes the
// least time (the rules are in hyperspot/ops), the loop of tile_loop.h.  What bounds
// it: 256 x 256 tiles power and the bytes on their way, 1.3 to 1.4 PFLOP/s with weights
// from memory, 1.45 where all loads are found in L2, 1.6 without loads; single waves
// some 9 us of start and end.  Non-temporal loads of w and tiles that begin at
// different columns are 2 to 8 % slower; 4 waves of 128 x 128 as fast.
//
// us, what was there (mostly the library's product, its pass or its norm) and here:
// silu(gate) * up 28672 x 4096 300 rows 85 79, 512 109 109 (but 6 less in the step),
// 880 197 187, 14336 x 2048 600 48 40, 2600 181 143; 4096 x 14336 with the norm 262 rows
// 64 52, 600 121 80, 1000 145 114, 7411 without 1006 647; 2048 x 7168, 600 rows 38 32.
// The library is faster for thousands of rows of full waves (8192 of 4096 x 14336 605
// 690).
#include <algorithm>

#include "tile_loop.h"

namespace {

constexpr int DIES = 8, TOGETHER = 8;

struct Wide {
  bf16* out;
  float* part;                 // [splits, M, N] with splits > 1
  const bf16* x;
  const bf16* w;
  int M, N, K;
  long xs, ws;                 // row strides
  int mt, nt, splits;          // tiles of rows, of outputs, parts of K
};

// H blocks of 32 rows of x, BN rows of w; the waves as in experts_tiles.hip.
template <int H, int MB, int BN, bool GATED>
DEV void wide_tile(const Wide& a, char* lds, int first_block, int m0, int n0, int z) {
  constexpr int BM = H * 32, OUT = GATED ? BN / 2 : BN;
  constexpr int NB = BN / 32, LW = BN / 64;
  using Loop = RingLoop<BM, BN, MB, NB, MB, LW, false>;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wid & 1;
  const int x_row = first_block * 32 + (wid >> 1 & 1) * (MB * 16);
  const int outs = GATED ? a.N >> 1 : a.N;
  const int all = a.K / 64;
  const int first = (int)((long)all * z / a.splits);
  const int chunks = (int)((long)all * (z + 1) / a.splits) - first;
  const RowLoads x_rows(a.x + m0 * a.xs + first * 64);
  const RowLoads w_rows(a.w + n0 * a.ws + first * 64);
  // this lane's 16 bytes of row lane / 8 of each 1-KB load; rows past the end
  // are the last one
  unsigned x_off[MB], w_off[LW];
  #pragma unroll
  for (int j = 0; j < MB; ++j) {
    const int r = first_block * 32 + ((wid & 3) * MB + j) * 8 + (lane >> 3);
    x_off[j] = (unsigned)(min(r, a.M - 1 - m0) * a.xs * 2) +
               ((lane & 7) ^ (r >> 1 & 7)) * 16;
  }
  #pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int r = (wid * LW + j) * 8 + (lane >> 3);
    const int n = min(GATED ? gated_row(r, 0) : plain_row(r), outs - 1 - n0) +
                  (GATED && r & 16 ? outs : 0);
    w_off[j] = (unsigned)(n * a.ws * 2) + ((lane & 7) ^ (r >> 1 & 7)) * 16;
  }
  Loop loop;
  loop.run(lds, x_row, part * (BN / 2), chunks, true,
           [&](char* l, int d, int i) {
             x_rows.to_lds(l + (first_block * 4 + (wid & 3) * MB + i) * 1024,
                           x_off[i], d * 128);
           },
           [&](char* l, int d, int i) {
             w_rows.to_lds(l + (wid * LW + i) * 1024, w_off[i], d * 128);
           });
  const int c0 = n0 + part * (OUT / 2);
  #pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int row = m0 + x_row + m * 16 + (lane & 15);
    if (row >= a.M) continue;
    if (a.splits > 1)
      store_part(loop.acc, m, a.part + ((long)z * a.M + row) * a.N + c0,
                 a.N - c0);
    else
      store_row<GATED>(loop.acc, m, a.out + (long)row * outs + c0, outs - c0);
  }
}

template <int H, int BN, bool GATED>
__global__ __launch_bounds__(512, 2) void gemm_wide_kernel(Wide a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  // Tiles in order: parts, groups of TOGETHER tiles of rows, tiles of outputs, the
  // tiles of a group.  Workgroups go to the dies in turn, and a die has neighbours in
  // this order, which share w and x.
  const int tiles = a.mt * a.nt * a.splits;
  const int die = blockIdx.x % DIES, from = (int)((long)tiles * die / DIES);
  int t = from + blockIdx.x / DIES;
  if (t >= (int)((long)tiles * (die + 1) / DIES)) return;
  const int z = t / (a.mt * a.nt);
  t -= z * a.mt * a.nt;
  const int g = t / (TOGETHER * a.nt), high = min(TOGETHER, a.mt - g * TOGETHER);
  t -= g * TOGETHER * a.nt;
  const int m0 = (g * TOGETHER + t % high) * (H * 32);
  const int n0 = t / high * (GATED ? BN / 2 : BN);
  // an even H has one code for all waves: what is read from memory for the first time
  // is waited for, code as well
  const bool later = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= 4;
  if (H % 2 == 0 || !later)
    wide_tile<H, H - H / 2, BN, GATED>(a, lds, later ? H / 2 : 0, m0, n0, z);
  else
    wide_tile<H, H / 2, BN, GATED>(a, lds, H - H / 2, m0, n0, z);
}

}  // namespace

// Tiles of 32 * high rows of x, high 4 to 8, by bn rows of w, 128 or 256.  Rows of x
// and w 16-byte aligned, K a multiple of 64, N of 8 (gated: 16), out contiguous;
// splits at most K / 64.  Without out the parts are left for the norm that adds them.
void launch_gemm_wide(bf16* out, float* part, const bf16* x, const bf16* w, int M,
                      int N, int K, long xs, long ws, int high, int bn, int splits,
                      bool gated, hipStream_t stream) {
  const int outs = gated ? bn / 2 : bn;
  Wide a{out, part, x, w, M, N, K, xs, ws, (M + high * 32 - 1) / (high * 32),
         ((gated ? N / 2 : N) + outs - 1) / outs, splits};
  const long tiles = (long)a.mt * a.nt * splits;
  const unsigned blocks = (unsigned)((tiles + DIES - 1) / DIES * DIES);
  #define RUN(H, BN, GATED)                                                 \
    {                                                                       \
      constexpr int XB = H * 32 * 128, WB = BN * 128;                       \
      constexpr int BYTES =                                                 \
          (3 * (XB + WB) <= 160 << 10 ? 3 : 2) * XB + 3 * WB;               \
      constexpr auto kernel = &gemm_wide_kernel<H, BN, GATED>;              \
      static const hipError_t set = hipFuncSetAttribute(                    \
          reinterpret_cast<const void*>(kernel),                            \
          hipFuncAttributeMaxDynamicSharedMemorySize, BYTES);               \
      HIP_CHECK(set);                                                       \
      kernel<<<blocks, 512, BYTES, stream>>>(a);                            \
    }
  #define KINDS(H)                                                          \
    case H:                                                                 \
      if (gated && bn == 256) RUN(H, 256, true)                             \
      else if (gated) RUN(H, 128, true)                                     \
      else if (bn == 256) RUN(H, 256, false)                                \
      else RUN(H, 128, false)                                               \
      break;
  switch (high) {
    KINDS(4) KINDS(5) KINDS(6) KINDS(7) KINDS(8)
    default: throw std::runtime_error("gemm_wide: 4 to 8 blocks of rows");
  }
  #undef KINDS
  #undef RUN
}
