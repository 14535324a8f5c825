// Fused NeoX-RoPE (q,k in place) + paged-KV append — one pass per token.
//
// The reference has no kernels (SURVEY.md §2.9 derives this list from the
// serving contract): rotating q/k and scattering k/v into the 288 GB-HBM3E
// paged pool in one kernel saves two extra passes over the qkv tensor every
// layer.  One 256-thread workgroup per token; cos/sin row staged in LDS.
#include "common.h"

// q: [T, H, D] bf16 (in place), k: [T, KV, D] (in place), v: [T, KV, D]
// cos_sin: [max_pos, D] float (cos | sin halves), positions: [T] i64
// slot_mapping: [T] i64 (slot = block*BS + off; <0 = no append)
// k_cache/v_cache: [NB, KV, BS, D] bf16
// q/k/v may be strided views into one fused qkv GEMM output buffer
// (token stride qs/ks/vs in elements; head dim contiguous).
// KV8: the paged cache stores OCP e4m3fn bytes (fp8 KV mode — halves the
// decode-attention HBM stream; scale fixed at 1.0, k/v magnitudes sit in
// the e4m3 normal range).
template <int D, bool KV8>
__global__ __launch_bounds__(256) void rope_kv_append_kernel(
    bf16* __restrict__ q, bf16* __restrict__ k, const bf16* __restrict__ v,
    const long* __restrict__ positions, const float* __restrict__ cos_sin,
    const long* __restrict__ slot_mapping, bf16* __restrict__ k_cache,
    bf16* __restrict__ v_cache, int H, int KV, int block_size,
    long qs_stride, long ks_stride, long vs_stride) {
  constexpr int HALF = D / 2;
  __shared__ float cs[D];
  const long t = blockIdx.x;
  const long pos = positions[t];
  const long slot = slot_mapping[t];
  const long blk = slot >= 0 ? slot / block_size : 0;
  const long off = slot >= 0 ? slot % block_size : 0;

  for (int i = threadIdx.x; i < D; i += 256)
    cs[i] = cos_sin[pos * D + i];
  __syncthreads();

  // rotate: thread u handles (head h, 2 consecutive pairs starting at 2j)
  // elements [2j, 2j+1] and [HALF+2j, HALF+2j+1] -> two ushort2 accesses
  const int PAIR2 = HALF / 2;               // u-slots per head
  const int total_q = H * PAIR2;
  for (int u = threadIdx.x; u < total_q; u += 256) {
    const int h = u / PAIR2, j = (u % PAIR2) * 2;
    bf16* base = q + t * qs_stride + h * D;
    ushort2 lo = *reinterpret_cast<ushort2*>(base + j);
    ushort2 hi = *reinterpret_cast<ushort2*>(base + HALF + j);
    float c0 = cs[j], c1 = cs[j + 1];
    float s0 = cs[HALF + j], s1 = cs[HALF + j + 1];
    float x0 = bf2f(lo.x), x1 = bf2f(lo.y);
    float y0 = bf2f(hi.x), y1 = bf2f(hi.y);
    lo.x = f2bf(x0 * c0 - y0 * s0); lo.y = f2bf(x1 * c1 - y1 * s1);
    hi.x = f2bf(y0 * c0 + x0 * s0); hi.y = f2bf(y1 * c1 + x1 * s1);
    *reinterpret_cast<ushort2*>(base + j) = lo;
    *reinterpret_cast<ushort2*>(base + HALF + j) = hi;
  }
  const int total_k = KV * PAIR2;
  for (int u = threadIdx.x; u < total_k; u += 256) {
    const int h = u / PAIR2, j = (u % PAIR2) * 2;
    bf16* base = k + t * ks_stride + h * D;
    ushort2 lo = *reinterpret_cast<ushort2*>(base + j);
    ushort2 hi = *reinterpret_cast<ushort2*>(base + HALF + j);
    float c0 = cs[j], c1 = cs[j + 1];
    float s0 = cs[HALF + j], s1 = cs[HALF + j + 1];
    float x0 = bf2f(lo.x), x1 = bf2f(lo.y);
    float y0 = bf2f(hi.x), y1 = bf2f(hi.y);
    const float r0 = x0 * c0 - y0 * s0, r1 = x1 * c1 - y1 * s1;
    const float r2 = y0 * c0 + x0 * s0, r3 = y1 * c1 + x1 * s1;
    lo.x = f2bf(r0); lo.y = f2bf(r1);
    hi.x = f2bf(r2); hi.y = f2bf(r3);
    *reinterpret_cast<ushort2*>(base + j) = lo;
    *reinterpret_cast<ushort2*>(base + HALF + j) = hi;
    if (slot >= 0) {
      if constexpr (KV8) {
        unsigned char* kc = reinterpret_cast<unsigned char*>(k_cache) +
            (((blk * KV + h) * block_size + off) * D);
        unsigned plo = __builtin_amdgcn_cvt_pk_fp8_f32(r0, r1, 0u, false);
        unsigned phi = __builtin_amdgcn_cvt_pk_fp8_f32(r2, r3, 0u, false);
        *reinterpret_cast<unsigned short*>(kc + j) = (unsigned short)plo;
        *reinterpret_cast<unsigned short*>(kc + HALF + j) =
            (unsigned short)phi;
      } else {
        bf16* kc = k_cache + (((blk * KV + h) * block_size + off) * D);
        *reinterpret_cast<ushort2*>(kc + j) = lo;
        *reinterpret_cast<ushort2*>(kc + HALF + j) = hi;
      }
    }
  }
  // v append: straight copy (bf16) or pack-to-fp8, 8-elem vectors
  if (slot >= 0) {
    const int total_v = KV * D / 8;
    for (int u = threadIdx.x; u < total_v; u += 256) {
      const int h = u / (D / 8), j = (u % (D / 8)) * 8;
      const bf16* src = v + t * vs_stride + h * D + j;
      if constexpr (KV8) {
        bf16x8 vv = load_bf16x8(src);
        unsigned w0 = 0, w1 = 0;
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(bf16x8_get(vv, 0),
                                             bf16x8_get(vv, 1), w0, false);
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(bf16x8_get(vv, 2),
                                             bf16x8_get(vv, 3), w0, true);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(bf16x8_get(vv, 4),
                                             bf16x8_get(vv, 5), w1, false);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(bf16x8_get(vv, 6),
                                             bf16x8_get(vv, 7), w1, true);
        uint2 pk{w0, w1};
        *reinterpret_cast<uint2*>(reinterpret_cast<unsigned char*>(v_cache)
            + (((blk * KV + h) * block_size + off) * D) + j) = pk;
      } else {
        bf16* vc = v_cache + (((blk * KV + h) * block_size + off) * D) + j;
        *reinterpret_cast<uint4*>(vc) =
            *reinterpret_cast<const uint4*>(src);
      }
    }
  }
}

// The same where q, k and the angles can be read 16 bytes at a time: 8 pairs a
// thread, whose angles it reads itself, so that a thread waits for one trip to memory
// and not for LDS and four small ones; the same bits.  What bounds it: memory, and with
// few rows that trip.  32 heads and 8 kv heads, us with 4 bytes a load and here: 128
// rows 4.5 3.5, 512 6.0 4.8, 2000 14.2 13.8, 8192 47.8 45.5, with e4m3 pages 45 42;
// 512 of 16 and 4 heads 4.8 3.9.
template <int D, bool KV8>
__global__ __launch_bounds__(256) void rope_kv_append8_kernel(
    bf16* __restrict__ q, bf16* __restrict__ k, const bf16* __restrict__ v,
    const long* __restrict__ positions, const float* __restrict__ cos_sin,
    const long* __restrict__ slot_mapping, bf16* __restrict__ k_cache,
    bf16* __restrict__ v_cache, int H, int KV, int block_size, long qs, long ks,
    long vs) {
  constexpr int HALF = D / 2, UNITS = HALF / 8;
  constexpr int ELEM = KV8 ? 1 : 2;
  const long t = blockIdx.x;
  const long slot = slot_mapping[t];
  const float* cs = cos_sin + positions[t] * D;
  const long blk = slot >= 0 ? slot / block_size : 0;
  const long off = slot >= 0 ? slot % block_size : 0;
  const int turned = (H + KV) * UNITS;         // then v, 8 elements a thread
  const int all = turned + (slot >= 0 ? KV * UNITS * 2 : 0);
  auto place = [&](bf16* cache, int h, int j) {
    return reinterpret_cast<char*>(cache) +
           (((blk * KV + h) * block_size + off) * D + j) * ELEM;
  };
  auto pack8 = [&](const float* r) {
    uint2 w{0, 0};
    w.x = __builtin_amdgcn_cvt_pk_fp8_f32(r[0], r[1], w.x, false);
    w.x = __builtin_amdgcn_cvt_pk_fp8_f32(r[2], r[3], w.x, true);
    w.y = __builtin_amdgcn_cvt_pk_fp8_f32(r[4], r[5], w.y, false);
    w.y = __builtin_amdgcn_cvt_pk_fp8_f32(r[6], r[7], w.y, true);
    return w;
  };
  for (int u = threadIdx.x; u < all; u += 256) {
    if (u >= turned) {
      const int w = u - turned, h = w / (UNITS * 2), j = w % (UNITS * 2) * 8;
      const bf16x8 x = load_bf16x8(v + t * vs + h * D + j);
      if constexpr (KV8) {
        float f[8];
        #pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = bf16x8_get(x, i);
        *reinterpret_cast<uint2*>(place(v_cache, h, j)) = pack8(f);
      } else {
        *reinterpret_cast<uint4*>(place(v_cache, h, j)) = x.raw;
      }
      continue;
    }
    const int h = u / UNITS, j = u % UNITS * 8;
    const bool key = h >= H;
    bf16* p = (key ? k + t * ks + (h - H) * D : q + t * qs + h * D) + j;
    bf16x8 lo = load_bf16x8(p), hi = load_bf16x8(p + HALF);
    f32x4_t c[2], s[2];
    #pragma unroll
    for (int i = 0; i < 2; ++i) {
      c[i] = *reinterpret_cast<const f32x4_t*>(cs + j + i * 4);
      s[i] = *reinterpret_cast<const f32x4_t*>(cs + HALF + j + i * 4);
    }
    float r[2][8];
    #pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = bf16x8_get(lo, i), y = bf16x8_get(hi, i);
      const float ci = c[i >> 2][i & 3], si = s[i >> 2][i & 3];
      r[0][i] = fmaf(x, ci, -(y * si));
      r[1][i] = fmaf(y, ci, x * si);
    }
    #pragma unroll
    for (int i = 0; i < 8; ++i) {
      bf16x8_set(lo, i, r[0][i]);
      bf16x8_set(hi, i, r[1][i]);
    }
    store_bf16x8(p, lo);
    store_bf16x8(p + HALF, hi);
    if (!key || slot < 0) continue;
    if constexpr (KV8) {
      *reinterpret_cast<uint2*>(place(k_cache, h - H, j)) = pack8(r[0]);
      *reinterpret_cast<uint2*>(place(k_cache, h - H, j + HALF)) = pack8(r[1]);
    } else {
      *reinterpret_cast<uint4*>(place(k_cache, h - H, j)) = lo.raw;
      *reinterpret_cast<uint4*>(place(k_cache, h - H, j + HALF)) = hi.raw;
    }
  }
}

void launch_rope_kv_append(bf16* q, bf16* k, const bf16* v,
                           const long* positions, const float* cos_sin,
                           const long* slot_mapping, bf16* k_cache,
                           bf16* v_cache, long T, int H, int KV, int D,
                           int block_size, long qs, long ks, long vs,
                           bool kv_fp8, hipStream_t stream) {
  const bool wide =
      qs % 8 == 0 && ks % 8 == 0 && vs % 8 == 0 &&
      ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
        reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(cos_sin) |
        reinterpret_cast<uintptr_t>(k_cache) |
        reinterpret_cast<uintptr_t>(v_cache)) & 15) == 0;
  #define RUN(KERNEL, D, KV8)                                               \
    KERNEL<D, KV8><<<(unsigned)T, 256, 0, stream>>>(                        \
        q, k, v, positions, cos_sin, slot_mapping, k_cache, v_cache, H, KV, \
        block_size, qs, ks, vs)
  #define EITHER(D, KV8)                                                    \
    if (wide) RUN(rope_kv_append8_kernel, D, KV8);                          \
    else RUN(rope_kv_append_kernel, D, KV8)
  if (D == 128 && kv_fp8) {
    EITHER(128, true);
  } else if (D == 128) {
    EITHER(128, false);
  } else if (D == 64 && !kv_fp8) {
    EITHER(64, false);
  } else {
    throw std::runtime_error("rope_kv_append: unsupported head_dim/dtype");
  }
  #undef EITHER
  #undef RUN
}

// Interleaved RoPE (dimension 2i with 2i+1, the first `rot` dimensions) and
// paged append for the windowed differential attention (csrc/attn_window.hip).
//
// q [T, NQ, D] rotates in place; k [T, NK, D] is rotated into the cache only.
// A kv head's maps are neighbours in k, so a cache row is MD = maps * D wide:
//   k_cache [NB, G, BS, MD]     v_cache [NB, G, E, BS]
// V pages are stored transposed: the attention kernels feed V^T tiles to the
// matrix cores straight from a page.  Angles p * freqs[i] are formed and
// reduced in double (freqs holds base^(-2i/rot)), so they stay exact to float
// rounding at any position without a table.
//
// V elements a thread at a time (1 or 8; 8 wants D, E, strides and bases in
// multiples of 8).  A workgroup takes TB neighbouring rows, blockIdx.y their q
// (0) or their k and v (1).  With TB > 1 tokens run fastest over the lanes of
// a V store, so the transposed writes of one sequence meet in the same page
// rows.
template <typename T, int V, int TB>
__global__ __launch_bounds__(256) void rope_pairs_append_kernel(
    T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
    const long* __restrict__ positions, const double* __restrict__ freqs,
    const long* __restrict__ slot_mapping, T* __restrict__ k_cache,
    T* __restrict__ v_cache, int NQ, int NK, int D, int G, int E, int rot,
    int block_size, long qs, long ks, long vs, long rows) {
  extern __shared__ float cs_all[];    // [TB][rot] (cos, sin) of each pair
  __shared__ long slot_of[TB];
  const long row0 = (long)blockIdx.x * TB;
  const int nrows = (int)min((long)TB, rows - row0);
  const int half = rot / 2;
  if (threadIdx.x < nrows)
    slot_of[threadIdx.x] = slot_mapping[row0 + threadIdx.x];
  for (int u = threadIdx.x; u < nrows * half; u += 256) {
    const int b = u / half, i = u % half;
    // angle in turns, reduced to [-1/2, 1/2]
    double a = (double)positions[row0 + b] * freqs[i] * 0.15915494309189535;
    a -= rint(a);
    float s, c;
    if constexpr (sizeof(T) == 2) {
      s = __builtin_amdgcn_sinf((float)a);       // argument in turns
      c = __builtin_amdgcn_cosf((float)a);
    } else {
      sincosf((float)(a * 6.283185307179586), &s, &c);
    }
    cs_all[b * rot + 2 * i] = c;
    cs_all[b * rot + 2 * i + 1] = s;
  }
  __syncthreads();
  // elements [d, d + W) of one head; W = V, or one pair where V = 1
  constexpr int W = V == 1 ? 2 : V;
  auto load = [&](const T* p, int d, float* x) {
    if constexpr (V == 1) {
      x[0] = Elem<T>::ld(p);
      x[1] = d + 1 < D ? Elem<T>::ld(p + 1) : 0.f;
    } else {
      #pragma unroll
      for (int i = 0; i < V; i += 4) load_vec<T, 4>(p + i, x + i);
    }
  };
  auto store = [&](T* p, int d, const float* x) {
    if constexpr (V == 1) {
      Elem<T>::st(p, x[0]);
      if (d + 1 < D) Elem<T>::st(p + 1, x[1]);
    } else {
      #pragma unroll
      for (int i = 0; i < V; i += 4) store_vec<T, 4>(p + i, x + i);
    }
  };
  auto rotate = [&](const float* cs, int d, float* x) {
    #pragma unroll
    for (int i = 0; i < W; i += 2)
      if (d + i < rot) {
        const float c = cs[d + i], s = cs[d + i + 1], u = x[i], w = x[i + 1];
        x[i] = u * c - w * s;
        x[i + 1] = w * c + u * s;
      }
  };
  const int nr = (rot + W - 1) / W;              // rotated chunks of a head
  if (blockIdx.y == 0) {
    for (int w = threadIdx.x; w < nrows * NQ * nr; w += 256) {
      const int b = w / (NQ * nr), u = w % (NQ * nr);
      const int h = u / nr, d = (u % nr) * W;
      T* p = q + (row0 + b) * qs + (long)h * D + d;
      float x[W];
      load(p, d, x);
      rotate(cs_all + b * rot, d, x);
      store(p, d, x);
    }
    return;
  }
  const int MD = NK / G * D;
  const int nd = (D + W - 1) / W;
  for (int w = threadIdx.x; w < nrows * NK * nd; w += 256) {
    const int b = w / (NK * nd), u = w % (NK * nd);
    const long slot = slot_of[b];
    if (slot < 0) continue;
    const long blk = slot / block_size, off = slot % block_size;
    const int h = u / nd, d = (u % nd) * W;
    const int g = h * D / MD, r = h * D - g * MD;
    float x[W];
    load(k + (row0 + b) * ks + (long)h * D + d, d, x);
    rotate(cs_all + b * rot, d, x);
    store(k_cache + ((blk * G + g) * block_size + off) * MD + r + d, d, x);
  }
  for (int w = threadIdx.x; w < TB * (G * E / V); w += 256) {
    const int b = w % TB, u = w / TB * V;
    if (b >= nrows || slot_of[b] < 0) continue;
    const long blk = slot_of[b] / block_size, off = slot_of[b] % block_size;
    T* vc = v_cache + (blk * G * E + u) * block_size + off;
    float x[V];
    #pragma unroll
    for (int i = 0; i < V; i += V == 1 ? 1 : 4)
      load_vec<T, V == 1 ? 1 : 4>(v + (row0 + b) * vs + u + i, x + i);
    #pragma unroll
    for (int i = 0; i < V; ++i) Elem<T>::st(vc + (long)i * block_size, x[i]);
  }
}

template <typename T>
void launch_rope_pairs_append(T* q, const T* k, const T* v,
                              const long* positions, const double* freqs,
                              const long* slot_mapping, T* k_cache,
                              T* v_cache, long rows, int NQ, int NK, int D,
                              int G, int E, int rot, int block_size, long qs,
                              long ks, long vs, hipStream_t stream) {
  if (rows == 0) return;
  auto aligned = [](const T* p) {
    return reinterpret_cast<uintptr_t>(p) % (8 * sizeof(T)) == 0;
  };
  const bool vec = D % 8 == 0 && E % 8 == 0 && qs % 8 == 0 && ks % 8 == 0 &&
                   vs % 8 == 0 && aligned(q) && aligned(k) && aligned(v);
  #define ROPE(V, TB)                                                       \
    rope_pairs_append_kernel<T, V, TB>                                      \
        <<<dim3((unsigned)((rows + TB - 1) / TB), 2), 256,                  \
           (TB * rot + 2) * sizeof(float), stream>>>(                       \
            q, k, v, positions, freqs, slot_mapping, k_cache, v_cache, NQ,  \
            NK, D, G, E, rot, block_size, qs, ks, vs, rows)
  if (!vec)
    ROPE(1, 1);
  else if (rows >= 4096 && rot <= 1024)
    ROPE(8, 8);
  else if (rows >= 1024 && rot <= 1024)
    ROPE(8, 4);
  else
    ROPE(8, 1);
  #undef ROPE
}
template void launch_rope_pairs_append<bf16>(
    bf16*, const bf16*, const bf16*, const long*, const double*, const long*,
    bf16*, bf16*, long, int, int, int, int, int, int, int, long, long, long,
    hipStream_t);
template void launch_rope_pairs_append<float>(
    float*, const float*, const float*, const long*, const double*,
    const long*, float*, float*, long, int, int, int, int, int, int, int,
    long, long, long, hipStream_t);
