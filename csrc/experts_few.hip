// Gated experts for few choices (gfx950), bf16, without a sort.
//
//   up    h[p, i] = silu(x[t] . w[e, i]) * (x[t] . w[e, N + i]) of choice p,
//         token t = p / div and expert e = ids[p]
//   down  y[p, n] = h[p] . w[e, n]
//
// What bounds it: the chosen experts' weights, read once.  A sort is a launch
// that everything waits for, and of a handful of choices every workgroup finds
// its own: it looks the expert numbers up, 64 a load, and has the choices of one
// expert as the columns of its products, 16 at a time, however few they are.
// Weights are the A operand of 16x16x32 products straight from memory; the waves
// divide K.  Of 16 rows of weights 8 are a gate's and 8 its up row's, so that
// there are twice as many workgroups as with 16 of each: those of the experts
// that are chosen spread over the compute units more evenly.
#include "common.h"

namespace {

constexpr int MOST = 384;            // choices

struct Few {
  bf16* out;
  int* place;                        // null, or of every choice: its number
  const bf16* x;
  const bf16* w;
  const int* ids;
  int P, E, N, K, div;
};

// WAVES divide K
template <int WAVES, bool UP>
__global__ __launch_bounds__(WAVES * 64) void experts_few_kernel(Few a) {
  constexpr int OUT = UP ? 8 : 16;
  __shared__ __attribute__((aligned(16))) float red[WAVES * 256];
  __shared__ int rows[WAVES][MOST];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, gr = lane >> 4;
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

  // rows of weights: gate and up rows in turn, 8 each
  const int n = n0 + (UP ? (col & 7) + (col & 8 ? a.N : 0) : col);
  const bf16* wp =
      a.w + ((long)e * (UP ? 2 * a.N : a.N) + n) * a.K + gr * 8;
  for (int r0 = 0; r0 < count; r0 += 16) {
    const bool live = r0 + col < count;
    const int choice = rows[wid][min(r0 + col, count - 1)];
    const bf16* xp = a.x + (long)(UP ? choice / a.div : choice) * a.K + gr * 8;
    f32x4_t acc = f32x4_t(0.f);
    #pragma unroll 2
    for (int k0 = wid * 64; k0 < a.K; k0 += WAVES * 64) {
      short8_t wf[2], xf[2];
      #pragma unroll
      for (int s = 0; s < 2; ++s) {
        wf[s] = *reinterpret_cast<const short8_t*>(wp + k0 + 32 * s);
        xf[s] = live ? *reinterpret_cast<const short8_t*>(xp + k0 + 32 * s)
                     : short8_t{};
      }
      #pragma unroll
      for (int s = 0; s < 2; ++s) acc = mfma16(wf[s], xf[s], acc);
    }
    if (r0) __syncthreads();
    *reinterpret_cast<f32x4_t*>(red + (wid * 64 + lane) * 4) = acc;
    __syncthreads();
    if (wid || !live || (UP && lane >= 32)) continue;
    auto total = [&](int l) {
      f32x4_t s = f32x4_t(0.f);
      #pragma unroll
      for (int v = 0; v < WAVES; ++v)
        s += *reinterpret_cast<const f32x4_t*>(red + (v * 64 + l) * 4);
      return s;
    };
    f32x4_t y = total(lane);
    if constexpr (UP) {
      const f32x4_t u = total(lane + 32);
      #pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = y[j] / (1.f + __expf(-y[j])) * u[j];
    }
    *reinterpret_cast<uint2*>(a.out + (long)choice * a.N + n0 + gr * 4) =
        uint2{cvt_pk_bf16(y[0], y[1]), cvt_pk_bf16(y[2], y[3])};
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
    experts_few_kernel<8, true>
        <<<dim3(N / 8, y), 512, 0, stream>>>(a);
  else
    experts_few_kernel<4, false>
        <<<dim3(N / 16, y), 256, 0, stream>>>(a);
}
