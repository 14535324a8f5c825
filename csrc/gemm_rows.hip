// out[M, N] = x[M, K] w[N, K]^T for few rows (gfx950), bf16 in and out, float
// sums; or e4m3 in, with scales of the rows, of which 16 bytes are two products'.
//
// What bounds it: reading w once.  So w is the A operand of 16x16x32 products
// straight from memory.  The rows of x, which every tile of w needs whole, go
// into LDS once a workgroup, and the workgroups stay: one or two a CU, each
// with every gridDim-th tile of up to 16 rows of w: of 12 or 8 where that
// spreads them better, whose loads the other lanes sit out.  (x from L2 beside
// every tile of w costs as many load instructions as w itself for each 16 rows:
// 28672 x 4096 took 50 us for one row and 72 us for 16.)  The 8 waves divide K,
// so that also a single tile has 8 KB of loads in flight a wave, and add up in
// LDS; the next tile's loads are issued before that.  x comes straight to LDS
// where K is a multiple of 512, otherwise 4 units of 16 bytes a thread at once
// (64 rows of 3904 x 384 12.4 -> 5.2 us, of 1760 x 768 12.8 -> 6.2, where each
// waited for the one before).
//
// A load has whole lines of w, 128 bytes of 8 rows, and is non-temporal: those do
// not hold a line of the unit's cache each while they wait, but what is left of
// half a line is read again.  An operand has 64 bytes of 16 rows, so two loads
// exchange halves.  Against loads of half lines, us: 1 row of 28672 x 4096 46 ->
// 39, of 4096 x 14336 27.5 -> 23, of 10240 x 4096 19.6 -> 16.5, of 2048 x 2048 4.5
// -> 4.2, 16 rows of 14336 x 2048 17.1 -> 14.3, 32 of 3072 x 2048 7.5 -> 7.0.
//
// us, library and here, weights from memory; and of tiles of 16 rows where others
// are taken (with loads of half lines):
//   28672 x 4096  1 row 64 39, 16 rows 66 42    4096 x 4096   1 15  9, 16 15 11
//   32768 x 4096  1 row 64 44, 16 rows 63 47    32768 x 2048  1 35 25, 32 37 29
//   12: 6144 x 4096  1 row 14.4 11.4 (14.5), 8 rows 14.4 13.2 (15.8)
//       3072 x 2048  1 row 11.2  5.0  (6.0), 32 rows 11.7 7.0 (8.2)
//       5120 x 4096  1 row 14.0 11.0 (13.7)
//   8: 2048 x 2048   1 row  8.7  4.2  (5.3), 32 rows 8.6 6.4 (7.5)
//      1536 x 4096   1 row 14.6  5.8  (7.9)
//      10240 x 4096  1 row 27.1 16.5 (21.0); 14336 x 2048 16.3 12.5 (14.8)
// e4m3, tiles of 64 x 32 and here: 6144 x 4096 1 row 9.8 6.8, 16 rows 11.1 8.9, 2048 x
// 2048 6.0 4.0 and 6.4 4.2; a decode step of 1 row, 4 wide layers, 405 -> 397.
#include <type_traits>

#include "common.h"

namespace {

constexpr int WAVES = 8;
constexpr int STEP = WAVES * 64;     // columns of a step of all waves
constexpr int U = 4;                 // steps a batch

struct Rows {
  bf16* out;
  const bf16* x;
  const bf16* w;
  int M, N, K;
  int rows;                          // of w a tile, at most 16
  long xs, ws, os;                   // row strides
  const float* x_scale;              // FP8: of a row of x, and of a row of w
  const float* w_scale;
};

// 16 bytes a lane, to the wave's LDS address + lane * 16
DEV void to_lds16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) unsigned*)g,
      (__attribute__((address_space(3))) unsigned*)l, 16, 0, 0);
}

// 32 products of a lane's 16 bytes, or 64 of e4m3
template <bool FP8>
DEV f32x4_t products_of(short8_t a, short8_t b, f32x4_t c) {
  if constexpr (!FP8) return mfma16(a, b, c);
  union { short8_t s; long d[2]; } x{a}, y{b};
  c = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(x.d[0], y.d[0], c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(x.d[1], y.d[1], c, 0, 0, 0);
}

// CT * 16 rows of x.  FP8: a column is two of e4m3
template <int CT, bool FP8>
__global__ __launch_bounds__(WAVES * 64, 4)
void gemm_rows_kernel(Rows a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* red = reinterpret_cast<float*>(smem);
  short* xl = reinterpret_cast<short*>(smem + WAVES * CT * 1024);
  const int xp = a.K + 8;            // row of x in LDS: 16 rows, 16 banks
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, gr = lane >> 4;
  const int at = gr * 16 + (col & 8);          // of a line's 64 columns
  const int tiles = (a.N + a.rows - 1) / a.rows;
  const int batches = (a.K + U * STEP - 1) / (U * STEP);

  short8_t wf[U][2], wn[U][2];
  auto fetch = [&](int tile, int batch) {
    const int k0 = batch * U * STEP + wid * 64;
    const bf16* p[2];
    #pragma unroll
    for (int s = 0; s < 2; ++s)
      p[s] = a.w +
             (long)min(tile * a.rows + s * 8 + (col & 7), a.N - 1) * a.ws + at;
    #pragma unroll
    for (int u = 0; u < U; ++u)
      #pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int k = k0 + u * STEP;
        wn[u][s] = k + at < a.K && s * 8 + (col & 7) < a.rows
            ? __builtin_nontemporal_load(
                  reinterpret_cast<const short8_t*>(p[s] + k))
            : short8_t{};
      }
  };
  int tile = blockIdx.x, batch = 0;
  fetch(tile, 0);
  if (a.K % 512 == 0) {              // a KB of a row a wave, straight to LDS
    const int parts = a.K / 512, n = a.M * parts;
    for (int i = wid; i < n; i += WAVES) {
      const int m = i / parts, c = (i - m * parts) * 512;
      to_lds16(a.x + m * a.xs + c + lane * 8, xl + m * xp + c);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {                           // 4 units of 16 bytes a thread at once
    constexpr int T = WAVES * 64;
    const int units = a.K / 8, n = a.M * units;
    for (int i = threadIdx.x; i < n; i += 4 * T) {
      short8_t v[4];
      int at[4];
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int u = min(i + j * T, n - 1);   // the last one again
        const int m = u / units, c = (u - m * units) * 8;
        v[j] = *reinterpret_cast<const short8_t*>(a.x + m * a.xs + c);
        at[j] = m * xp + c;
      }
      #pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<short8_t*>(xl + at[j]) = v[j];
    }
  }
  const short* xr[CT];
  #pragma unroll
  for (int t = 0; t < CT; ++t)       // rows past the end: not stored
    xr[t] = xl + min(t * 16 + col, a.M - 1) * xp + gr * 16;
  f32x4_t acc[CT];
  #pragma unroll
  for (int t = 0; t < CT; ++t) acc[t] = f32x4_t(0.f);
  __syncthreads();

  while (tile < tiles) {
    #pragma unroll
    for (int u = 0; u < U; ++u) {
      wf[u][0] = wn[u][0];
      wf[u][1] = wn[u][1];
      exchange_halves(wf[u][0], wf[u][1]);
    }
    const int k0 = batch * U * STEP + wid * 64, now = tile;
    if (++batch == batches) {
      batch = 0;
      tile += gridDim.x;
    }
    if (tile < tiles) fetch(tile, batch);
    auto products = [&](auto whole) {
      #pragma unroll
      for (int u = 0; u < U; ++u)
        #pragma unroll
        for (int s = 0; s < 2; ++s) {
          // columns past the end: x is zero as w is, for the last ones may
          // hold an infinity
          const int k = k0 + u * STEP + 8 * s;
          if (!whole && k >= a.K) continue;
          const bool in = whole || k + gr * 16 < a.K;
          #pragma unroll
          for (int t = 0; t < CT; ++t) {
            const short8_t v = *reinterpret_cast<const short8_t*>(
                xr[t] + (in ? k : 0));
            acc[t] = products_of<FP8>(wf[u][s], in ? v : short8_t{}, acc[t]);
          }
        }
    };
    if (k0 + (U - 1) * STEP + 64 <= a.K)
      products(std::true_type{});
    else
      products(std::false_type{});
    if (batch) continue;
    #pragma unroll
    for (int t = 0; t < CT; ++t) {
      *reinterpret_cast<f32x4_t*>(red + ((wid * CT + t) * 64 + lane) * 4) =
          acc[t];
      acc[t] = f32x4_t(0.f);
    }
    __syncthreads();
    if (wid < CT) {
      f32x4_t y = f32x4_t(0.f);
      #pragma unroll
      for (int v = 0; v < WAVES; ++v)
        y += *reinterpret_cast<const f32x4_t*>(
            red + ((v * CT + wid) * 64 + lane) * 4);
      const int n = now * a.rows + gr * 4, m = wid * 16 + col;
      if (m < a.M && n < a.N && gr * 4 < a.rows) {   // multiples of 4
        if constexpr (FP8) {
          const float xs = a.x_scale[m];
          const f32x4_t ws = *reinterpret_cast<const f32x4_t*>(a.w_scale + n);
          #pragma unroll
          for (int j = 0; j < 4; ++j) y[j] = y[j] * xs * ws[j];
        }
        *reinterpret_cast<uint2*>(a.out + m * a.os + n) =
            uint2{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3])};
      }
    }
    __syncthreads();
  }
}

constexpr int LDS = 160 * 1024;

// 16-row tiles of x a workgroup has
int row_tiles(int M) { return M <= 16 ? 1 : M <= 32 ? 2 : 4; }

int lds_bytes(int M, int K) {
  return WAVES * row_tiles(M) * 1024 + M * (K + 8) * 2;
}

// rows of w a tile: those that the busiest CU has are fewest
int tile_rows(int N) {
  int best = 16, least = 0;
  for (int rows = 16; rows >= 8; rows -= 4) {
    const int tiles = (N + rows - 1) / rows;
    const int most = (tiles + 255) / 256 * rows;
    if (least == 0 || most < least) {
      best = rows;
      least = most;
    }
  }
  return best;
}

}  // namespace

// whether M rows of K columns are taken
bool gemm_rows_fits(long M, long K) {
  return M >= 1 && M <= 64 && K >= 8 && K <= 65536 &&
         lds_bytes((int)M, (int)K) <= LDS;
}

// N a multiple of 4, K of 8; rows of x and w 16-byte, of out 8-byte aligned.  With
// scales x and w are e4m3, and K and their strides half of what they are
void launch_gemm_rows(bf16* out, const bf16* x, const bf16* w,
                      const float* x_scale, const float* w_scale, int M, int N,
                      int K, long xs, long ws, long os, hipStream_t stream) {
  const int rows = tile_rows(N);
  const Rows a{out, x, w, M, N, K, rows, xs, ws, os, x_scale, w_scale};
  const int lds = lds_bytes(M, K), tiles = (N + rows - 1) / rows;
  const int most = lds * 2 <= LDS ? 512 : 256;     // that a CU holds at once
  const unsigned grid = (unsigned)(tiles < most ? tiles : most);
  #define KIND(CT, FP8)                                                     \
    {                                                                       \
      static const hipError_t set = hipFuncSetAttribute(                    \
          reinterpret_cast<const void*>(&gemm_rows_kernel<CT, FP8>),        \
          hipFuncAttributeMaxDynamicSharedMemorySize, LDS);                 \
      HIP_CHECK(set);                                                       \
      gemm_rows_kernel<CT, FP8><<<grid, WAVES * 64, lds, stream>>>(a);      \
    }
  #define RUN(CT)                                                           \
    {                                                                       \
      if (x_scale) KIND(CT, true)                                           \
      else KIND(CT, false)                                                  \
    }
  switch (row_tiles(M)) {
    case 1: RUN(1) break;
    case 2: RUN(2) break;
    default: RUN(4)
  }
  #undef RUN
  #undef KIND
}
