// Gated experts for few choices (gfx950), bf16, without a sort.
//
//   up    h[p, i] = silu(x[t] . w[e, i]) * (x[t] . w[e, N + i]) of choice p,
//         token t = p / div and expert e = ids[p]
//   down  y[p, n] = h[p] . w[e, n]
//
// What bounds it: the chosen experts' weights, read once.  A sort is a launch
// that everything waits for, and of a handful of choices every workgroup finds
// its own: it looks the expert numbers up, 64 a load, and has the choices of one
// expert as the columns of its products, however few they are.  A workgroup has
// 16 rows of weights, 8 of a gate and 8 of its up row or 16 in turn, so that the
// chosen experts spread over the compute units evenly; its waves divide K.
//
// Weights are the A operand of 16x16x32 products straight from memory, and a
// load takes whole lines of them, 128 bytes of 8 rows, non-temporal: those do
// not hold a line of the unit's cache each while they wait, but two loads of
// half a line would read it twice.  So row i of A is the first half of a line
// of 8 rows, row 8 + i its second half; the columns of B are the halves of the
// lines of 8 choices likewise, and of a product the two squares count where the
// halves are the same.  us, up and down, and with halves of 16 lines a load (not
// non-temporal; that was slower still):
//   32 experts of 1024 x 2048, 4 each   1 row 9.0 5.8 (10.1 7.2), 4 rows 22.7
//     12.9 (25.5 14.4), 16 rows 44 24 (49 27)
//   8 experts of 14336 x 4096, 2 each   1 row 75 40 (82 59), 4 rows 175 92
//     (200 125), 10 rows 242 138 (302 177)
#include <type_traits>

#include "common.h"

namespace {

constexpr int MOST = 384;            // choices
constexpr int WAVES = 4;             // divide K
constexpr int STEP = WAVES * 64;     // columns of a step of all waves

struct Few {
  bf16* out;
  int* place;                        // null, or of every choice: its number
  const bf16* x;
  const bf16* w;
  const int* ids;
  int P, E, N, K, div;
};

template <bool UP>
__global__ __launch_bounds__(WAVES * 64) void experts_few_kernel(Few a) {
  constexpr int OUT = UP ? 8 : 16;
  __shared__ f32x4_t red[WAVES][2][2][16];     // rows of 8, halves, 4 rows of 1
  __shared__ int rows[WAVES][MOST];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 7, half = lane >> 3 & 1, gr = lane >> 4;
  const int n0 = blockIdx.x * OUT;
  if (a.place && blockIdx.x == 0 && blockIdx.y == 0)
    for (int p = threadIdx.x; p < a.P; p += WAVES * 64)
      a.place[p] = (unsigned)a.ids[p] < (unsigned)a.E ? p : -1;
  // as many experts as choices at most: the choices' own, each where it is
  // named first; otherwise all of them
  int e = blockIdx.y;
  const bool named = a.P <= a.E;     // at most 64
  if (named) e = a.ids[e];
  if (e < 0 || e >= a.E) return;
  int count = 0;
  for (int p0 = 0; p0 < a.P; p0 += 64) {
    const int p = p0 + lane;
    const unsigned long long has =
        __ballot(p < a.P && a.ids[min(p, a.P - 1)] == e);
    if (named && __ffsll(has) - 1 != (int)blockIdx.y) return;
    if (has >> lane & 1)
      rows[wid][count + __popcll(has & ((1ull << lane) - 1))] = p;
    count += __popcll(has);
  }
  if (count == 0) return;

  const int at = half * 32 + gr * 8;           // a lane's part of a line
  const bf16* wp =
      a.w + ((long)e * (UP ? 2 * a.N : a.N) + n0 + col) * a.K + at;
  const long next = (long)(UP ? a.N : 8) * a.K;    // up rows, or 8 rows on
  // Workgroups begin at different columns where rows are multiples of 4 KB, of
  // which one column is a few channels of memory; by their rows of weights, so
  // that a choice's sums do not depend on the others.  us, up and down: 8 experts of
  // 14336 x 4096, 2 choices 79.3 43.8 -> 74.4 39.9, 16 258 145 -> 247 133; 16 of 2048
  // x 4096, 8 48.1 26.7 -> 44.4 23.3; of 3072 x 6144, 88.2 -> 86.5 (up).  Of other
  // lengths it is 0 to 2 % slower, and even where the up product has rows of 4 KB: 32 of
  // 1024 x 2048, 16 21.7 21.9, 64 of 1408 x 2048, 24 42.1 41.1.
  const int batches = a.K / (2 * STEP);
  const int begin = a.K % 2048 == 0 && a.K > (UP ? 2048 : 0)
      ? (int)(blockIdx.x / 8 % (unsigned)batches) : 0;
  for (int r0 = 0; r0 < count; r0 += 16) {
    const bf16* xp[2];                         // of 8 choices and 8 more
    bool live[2];
    #pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int r = r0 + g * 8 + col;
      live[g] = r < count;
      const int choice = rows[wid][min(r, count - 1)];
      xp[g] = a.x + (long)(UP ? choice / a.div : choice) * a.K + at;
    }
    const bool more = r0 + 8 < count;
    f32x4_t acc[2][2];
    #pragma unroll
    for (int i = 0; i < 4; ++i) acc[i >> 1][i & 1] = f32x4_t(0.f);
    auto products = [&](int k, auto steps) {
      constexpr int S = decltype(steps)::value;
      short8_t wf[S][2], xf[S];
      #pragma unroll
      for (int u = 0; u < S; ++u)
        #pragma unroll
        for (int s = 0; s < 2; ++s)
          wf[u][s] = __builtin_nontemporal_load(
              reinterpret_cast<const short8_t*>(wp + s * next + k + u * STEP));
      auto add = [&](int g) {
        #pragma unroll
        for (int u = 0; u < S; ++u)
          xf[u] = live[g] ? *reinterpret_cast<const short8_t*>(
                                xp[g] + k + u * STEP)
                          : short8_t{};
        #pragma unroll
        for (int u = 0; u < S; ++u)
          #pragma unroll
          for (int s = 0; s < 2; ++s)
            acc[g][s] = mfma16(wf[u][s], xf[u], acc[g][s]);
      };
      add(0);
      if (more) add(1);
    };
    int turn = begin;
    #pragma unroll 1
    for (int i = 0; i < batches; ++i) {
      products(turn * 2 * STEP + wid * 64, std::integral_constant<int, 2>{});
      if (++turn == batches) turn = 0;
    }
    for (int k = batches * 2 * STEP + wid * 64; k < a.K; k += STEP)
      products(k, std::integral_constant<int, 1>{});

    #pragma unroll
    for (int g = 0; g < 2; ++g) {
      if (g && !more) break;
      if (r0 || g) __syncthreads();
      if (half == gr >> 1)
        #pragma unroll
        for (int s = 0; s < 2; ++s)
          red[wid][s][half][(gr & 1) * 8 + col] = acc[g][s];
      __syncthreads();
      if (wid) continue;
      // lane: half, 8 rows, 4 rows of them, choice
      f32x4_t y = f32x4_t(0.f);
      #pragma unroll
      for (int v = 0; v < WAVES; ++v)
        y += red[v][lane >> 4 & 1][lane >> 5][lane & 15];
      #pragma unroll
      for (int j = 0; j < 4; ++j) y[j] += __shfl_xor(y[j], 32);
      if constexpr (UP)
        #pragma unroll
        for (int j = 0; j < 4; ++j)
          y[j] = y[j] / (1.f + __expf(-y[j])) * __shfl_xor(y[j], 16);
      if (!live[g] || lane >= (UP ? 16 : 32)) continue;
      *reinterpret_cast<uint2*>(a.out +
                                (long)rows[0][r0 + g * 8 + col] * a.N + n0 +
                                (lane >> 3) * 4) =
          uint2{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3])};
    }
  }
}

}  // namespace

// P choices, 1 to 384, of 64 experts at most; N and K multiples of 128;
// everything contiguous
void launch_experts_few(bool up, bf16* out, int* place, const bf16* x,
                        const bf16* w, const int* ids, int P, int E, int N,
                        int K, int div, hipStream_t stream) {
  const Few a{out, place, x, w, ids, P, E, N, K, div};
  const int y = P < E ? P : E;
  if (up)
    experts_few_kernel<true><<<dim3(N / 8, y), WAVES * 64, 0, stream>>>(a);
  else
    experts_few_kernel<false><<<dim3(N / 16, y), WAVES * 64, 0, stream>>>(a);
}
