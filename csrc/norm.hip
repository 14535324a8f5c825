// RMSNorm + fused residual-add RMSNorm, bf16, row-per-workgroup.
//
// What bounds it: many rows, memory (8192 rows of 4096 at 6.5 TB/s); few, the
// trips to memory one after the other, so that all loads of a row, the weights
// among them, are issued before anything waits (us for 1, 32, 256 rows of 4096
// 2.7 3.0 3.4 when each waited for the one before, 2.4 2.5 3.1 so; of 8192 3.7
// 4.0 5.0 and 3.2 3.4 4.6).  One 256-thread workgroup per token row, bf16x8
// vector loads (scalar bf16 loads are ~2x slower), fp32 accumulation, row held
// in registers between the sumsq pass and the scale pass so each byte is read
// once.
#include "common.h"

// CH * 256 threads * 8 elements hold a row
template <int CH>
__global__ __launch_bounds__(256) void rmsnorm_kernel(
    bf16* __restrict__ out, const bf16* __restrict__ x,
    const bf16* __restrict__ w, float eps, int hidden) {
  __shared__ float scratch[4];
  const long row = blockIdx.x;
  const bf16* xr = x + row * (long)hidden;
  bf16* orow = out + row * (long)hidden;

  bf16x8 v[CH], wv[CH];
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      v[c] = load_bf16x8(xr + base);
      wv[c] = load_bf16x8(w + base);
    }
  }
  float ss = 0.f;
  #pragma unroll
  for (int c = 0; c < CH; ++c)
    if ((c * 256 + threadIdx.x) * 8 < hidden) {
      #pragma unroll
      for (int i = 0; i < 8; ++i) {
        float f = bf16x8_get(v[c], i);
        ss += f * f;
      }
    }
  const float total = block_reduce_sum_256(ss, scratch);
  const float rs = rsqrtf(total / hidden + eps);
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      bf16x8 o;
      #pragma unroll
      for (int i = 0; i < 8; ++i)
        bf16x8_set(o, i, bf16x8_get(v[c], i) * rs * bf16x8_get(wv[c], i));
      store_bf16x8(orow + base, o);
    }
  }
}

// x <- rmsnorm(residual + x) * w ; residual <- residual + x   (both in place)
template <int CH>
__global__ __launch_bounds__(256) void fused_add_rmsnorm_kernel(
    bf16* __restrict__ x, bf16* __restrict__ residual,
    const bf16* __restrict__ w, float eps, int hidden) {
  __shared__ float scratch[4];
  const long row = blockIdx.x;
  bf16* xr = x + row * (long)hidden;
  bf16* rr = residual + row * (long)hidden;

  bf16x8 xv[CH], rv[CH], wv[CH];
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      xv[c] = load_bf16x8(xr + base);
      rv[c] = load_bf16x8(rr + base);
      wv[c] = load_bf16x8(w + base);
    }
  }
  float r[CH][8];
  float ss = 0.f;
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      bf16x8 o;
      #pragma unroll
      for (int i = 0; i < 8; ++i) {
        float f = bf16x8_get(xv[c], i) + bf16x8_get(rv[c], i);
        r[c][i] = f;
        ss += f * f;
        bf16x8_set(o, i, f);
      }
      store_bf16x8(rr + base, o);   // new residual
    }
  }
  const float total = block_reduce_sum_256(ss, scratch);
  const float rs = rsqrtf(total / hidden + eps);
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      bf16x8 o;
      #pragma unroll
      for (int i = 0; i < 8; ++i)
        bf16x8_set(o, i, r[c][i] * rs * bf16x8_get(wv[c], i));
      store_bf16x8(xr + base, o);
    }
  }
}

// x <- rmsnorm(residual + y) * w ; residual <- residual + y, where y is the sum
// of `parts` float products [parts, rows, hidden], rounded as a product is.
// Adding them up here saves a launch and a trip to memory: us of product and
// norm, 32 rows of 2048 x 7168 in 8 parts 14.2 -> 13.3, 256 of 4096 x 4096 in 2
// 27.1 -> 24.3, 256 of 4096 x 14336 in 4 55 -> 51.5 (32 rows in 8, 29.6 29.8).
template <int CH>
__global__ __launch_bounds__(256) void parts_add_rmsnorm_kernel(
    bf16* __restrict__ x, const float* __restrict__ part, int parts,
    bf16* __restrict__ residual, const bf16* __restrict__ w, float eps,
    int hidden) {
  __shared__ float scratch[4];
  const long row = blockIdx.x;
  const long stride = (long)gridDim.x * hidden;     // of a part
  bf16* xr = x + row * (long)hidden;
  bf16* rr = residual + row * (long)hidden;

  bf16x8 rv[CH], wv[CH];
  f32x4_t y[CH][2];
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      rv[c] = load_bf16x8(rr + base);
      wv[c] = load_bf16x8(w + base);
      const float* p = part + row * hidden + base;
      y[c][0] = *reinterpret_cast<const f32x4_t*>(p);
      y[c][1] = *reinterpret_cast<const f32x4_t*>(p + 4);
      #pragma unroll 4
      for (int z = 1; z < parts; ++z) {
        y[c][0] += *reinterpret_cast<const f32x4_t*>(p + z * stride);
        y[c][1] += *reinterpret_cast<const f32x4_t*>(p + z * stride + 4);
      }
    }
  }
  float r[CH][8];
  float ss = 0.f;
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      bf16x8 o;
      #pragma unroll
      for (int i = 0; i < 8; ++i) {
        float f = bf2f(f2bf(y[c][i >> 2][i & 3])) + bf16x8_get(rv[c], i);
        r[c][i] = f;
        ss += f * f;
        bf16x8_set(o, i, f);
      }
      store_bf16x8(rr + base, o);   // new residual
    }
  }
  const float total = block_reduce_sum_256(ss, scratch);
  const float rs = rsqrtf(total / hidden + eps);
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      bf16x8 o;
      #pragma unroll
      for (int i = 0; i < 8; ++i)
        bf16x8_set(o, i, r[c][i] * rs * bf16x8_get(wv[c], i));
      store_bf16x8(xr + base, o);
    }
  }
}

// x <- rmsnorm(residual + y) * w ; residual <- residual + y, where y is the
// weighted sum of a row's n choices, rounded as it would be on its own: weight
// [row, k] * data[place[row, k]] (place -1: nothing).  A launch and a trip to
// memory less than the sum and the norm; the choices' rows are loaded 4 at a time
// beside the rest.
// us of both and of one: 4 rows of 2048, 4 choices 5.9 -> 3.1; 192 of 4096, 2
// choices 7.4 -> 3.7; 2000 of them 22 -> 13; 8000 75 -> 48.
template <int CH>
__global__ __launch_bounds__(256) void choices_add_rmsnorm_kernel(
    bf16* __restrict__ x, const bf16* __restrict__ data,
    const int* __restrict__ place, const float* __restrict__ weight, int n,
    bf16* __restrict__ residual, const bf16* __restrict__ w, float eps,
    int hidden) {
  __shared__ float scratch[4];
  const long row = blockIdx.x;
  bf16* xr = x + row * (long)hidden;
  bf16* rr = residual + row * (long)hidden;

  bf16x8 rv[CH], wv[CH];
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      rv[c] = load_bf16x8(rr + base);
      wv[c] = load_bf16x8(w + base);
    }
  }
  float r[CH][8];
  #pragma unroll
  for (int c = 0; c < CH; ++c)
    #pragma unroll
    for (int i = 0; i < 8; ++i) r[c][i] = 0.f;
  for (int k0 = 0; k0 < n; k0 += 4) {
    long from[4];
    float share[4];
    #pragma unroll
    for (int k = 0; k < 4; ++k) {
      const long i = row * n + min(k0 + k, n - 1);
      from[k] = k0 + k < n ? place[i] : -1;
      share[k] = weight[i];
    }
    bf16x8 yv[4][CH];
    #pragma unroll
    for (int k = 0; k < 4; ++k)
      #pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int base = (c * 256 + threadIdx.x) * 8;
        if (from[k] >= 0 && base < hidden)
          yv[k][c] = load_bf16x8(data + from[k] * hidden + base);
      }
    #pragma unroll
    for (int k = 0; k < 4; ++k)
      if (from[k] >= 0) {
        #pragma unroll
        for (int c = 0; c < CH; ++c)
          #pragma unroll
          for (int i = 0; i < 8; ++i)
            r[c][i] += share[k] * bf16x8_get(yv[k][c], i);
      }
  }
  float ss = 0.f;
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      bf16x8 o;
      #pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float f = bf2f(f2bf(r[c][i])) + bf16x8_get(rv[c], i);
        r[c][i] = f;
        ss += f * f;
        bf16x8_set(o, i, f);
      }
      store_bf16x8(rr + base, o);   // new residual
    }
  }
  const float total = block_reduce_sum_256(ss, scratch);
  const float rs = rsqrtf(total / hidden + eps);
  #pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int base = (c * 256 + threadIdx.x) * 8;
    if (base < hidden) {
      bf16x8 o;
      #pragma unroll
      for (int i = 0; i < 8; ++i)
        bf16x8_set(o, i, r[c][i] * rs * bf16x8_get(wv[c], i));
      store_bf16x8(xr + base, o);
    }
  }
}

// chunks that hold a row of up to 4096, 8192 or 16384 elements
static int chunks(int hidden) {
  return hidden <= 4096 ? 2 : hidden <= 8192 ? 4 : 8;
}

void launch_rmsnorm(bf16* out, const bf16* x, const bf16* w, float eps,
                    long rows, int hidden, hipStream_t stream) {
  const auto kernel = chunks(hidden) == 2   ? rmsnorm_kernel<2>
                      : chunks(hidden) == 4 ? rmsnorm_kernel<4>
                                            : rmsnorm_kernel<8>;
  kernel<<<dim3((unsigned)rows), dim3(256), 0, stream>>>(out, x, w, eps,
                                                         hidden);
}

void launch_fused_add_rmsnorm(bf16* x, bf16* residual, const bf16* w,
                              float eps, long rows, int hidden,
                              hipStream_t stream) {
  const auto kernel = chunks(hidden) == 2   ? fused_add_rmsnorm_kernel<2>
                      : chunks(hidden) == 4 ? fused_add_rmsnorm_kernel<4>
                                            : fused_add_rmsnorm_kernel<8>;
  kernel<<<dim3((unsigned)rows), dim3(256), 0, stream>>>(x, residual, w, eps,
                                                         hidden);
}

// 2 to 8 parts, hidden at most 8192
void launch_parts_add_rmsnorm(bf16* x, const float* part, int parts,
                              bf16* residual, const bf16* w, float eps,
                              long rows, int hidden, hipStream_t stream) {
  const auto kernel = hidden <= 2048   ? parts_add_rmsnorm_kernel<1>
                      : hidden <= 4096 ? parts_add_rmsnorm_kernel<2>
                                       : parts_add_rmsnorm_kernel<4>;
  kernel<<<dim3((unsigned)rows), dim3(256), 0, stream>>>(
      x, part, parts, residual, w, eps, hidden);
}

// hidden at most 8192
void launch_choices_add_rmsnorm(bf16* x, const bf16* data, const int* place,
                                const float* weight, int n, bf16* residual,
                                const bf16* w, float eps, long rows,
                                int hidden, hipStream_t stream) {
  const auto kernel = hidden <= 2048   ? choices_add_rmsnorm_kernel<1>
                      : hidden <= 4096 ? choices_add_rmsnorm_kernel<2>
                                       : choices_add_rmsnorm_kernel<4>;
  kernel<<<dim3((unsigned)rows), dim3(256), 0, stream>>>(
      x, data, place, weight, n, residual, w, eps, hidden);
}
