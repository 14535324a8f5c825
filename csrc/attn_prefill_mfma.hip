// Causal prompt attention on the matrix cores (gfx950), bf16, head_dim 128.
//
// Sequence s has the rows seq_start[s] .. seq_start[s + 1] of q; row i of it
// sees the first before + i + 1 tokens.  Three places that keys and values
// come from:
//   ROWS    k and v beside q: whole prompts, before = 0
//   PAGES   the bf16 pages: portions whose earlier tokens are cached,
//           before = ctx_lens[first row] - 1
//   PAGES8  the same with e4m3 pages
//
// What bounds it: the matrix products, 4 * 128 operations a score, against
// about as many cycles of vector work (exponential, maximum, sum,
// conversion).  So: scores are formed transposed, S^T = K Q^T, with the K row
// that feeds matrix row i permuted so that the scores a lane holds are 8
// consecutive tokens of one query row, which is the operand P^T of
// O^T = V^T P^T: weights never leave their registers, and the running maximum
// and its rescaling are one value a lane.  The rescaling is left out while no
// row's maximum grew (pages: by more than 2^GROW).  V^T is read with the
// transposing LDS load.
//
// A workgroup is 4 waves of 32 rows: HG heads of one kv head share a tile of
// 64 tokens, so that the causal edge of 4 heads costs 32 rows of work and not
// 128.  Tiles are double-buffered and (bf16) go from memory to LDS directly,
// 16 bytes a lane; 64 KB of LDS and 256 registers leave two workgroups a CU,
// whose products and vector work overlap.  Heads vary fastest over the
// workgroups: with 8 kv heads a die has one of them, and its keys and values
// stay in the die's L2.  Later rows see more and start first.
//
// Within a tile the operands of 8 products are loaded ahead of them, and the next
// 16 tokens' weights are formed between the products of the last 16, not before
// them.  Tiles come by buffer loads: beside loads from a global address to LDS
// the compiler waited for all LDS reads wherever it needed the oldest.  Long
// prompts are bound by power: with zeros as data 7808 rows after 8192 cached
// tokens take 1.86 ms, with normal values 2.47.
//
// 32 heads, 8 kv heads, us without those two steps and now: a prompt of 8192
// tokens 612 601 (915 TFLOP/s), of 512 18.6 17.8, 8 of 1000 124 122; 7808 tokens
// after 8192 cached ones 2587 2487, of e4m3 2630 2592, 500 after 500 39 34.
// Weights that went through LDS and tiles of 256 rows of one head took 3.6 times
// as long for 8192 tokens, one workgroup a row 37.6 ms for 7808 after 8192.
//
// ROWS: weights are rounded to bf16, relative to the maximum after each tile of
// 64 tokens, and summed in a fixed order.  Both are a part of the result: a
// model with 8-bit activations rounds it to few steps again, and a last bit
// decides between two of them.  Pages: the weights are floats in the
// row-by-row kernel, so they enter as three parts, which hold the 24 bits of a
// float; two were off by up to 2^-20 of what they weigh (and took 2.07 ms).
#include <float.h>

#include "tile_loop.h"

namespace {

constexpr int HD = 128;
constexpr int KV = 64;            // tokens of a tile
constexpr int WAVE_ROWS = 32;
constexpr int PAGE = 16;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float GROW = 8.f;
enum Source { ROWS, PAGES, PAGES8 };
enum { VALU = 0x002, PRODUCT = 0x008, DS_READ = 0x100 };  // for the scheduler

typedef __attribute__((ext_vector_type(4))) short short4_t;
typedef __attribute__((ext_vector_type(2))) float float2_t;

struct Prefill {
  bf16* out;
  const bf16* q;
  const bf16* k;             // rows, or pages
  const bf16* v;
  const int* seq_start;
  const int* ctx_lens;       // pages only
  const int* block_tables;
  int seqs, H, G, max_blocks, min_rows;
  float scale;               // positive: its sign, or a scale of zero, is
  short q_and, q_xor;        // applied to the bits of q; pages: times log2(e)
  long sq, sk, sv;           // strides of a row
};

DEV float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// four rows of one column: in every 16 lanes, lane i passes the address of
// row i / 4, columns 4 (i % 4), and receives column i
DEV short4_t lds_read_tr(const short* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) short4_t*)p);
}

// not to become a part of a fused operation
DEV float product(float x, float y) {
  #pragma clang fp contract(off)
  return x * y;
}

// x of the upper half of the lanes against y of the lower
DEV void swap_halves(float& x, float& y) {
  const auto r = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r[0]);
  y = __uint_as_float(r[1]);
}

// of the lanes i and i ^ 32
DEV float max_halves(float x) {
  const unsigned u = __float_as_uint(x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// 16-byte unit c of row r of a tile in LDS (rows of 16 units): the reads of
// 16 rows of one unit, and of 4 rows of 64 bytes each, spread over the banks
DEV int k_unit(int r, int c) { return r * 16 + (c ^ (r & 15)); }
DEV int v_unit(int r, int c) { return r * 16 + (c ^ (r & 3) << 2); }

// 4 e4m3 bytes as bf16, exactly
DEV uint2 widen(unsigned x) {
  const float2_t a = __builtin_amdgcn_cvt_pk_f32_fp8(x, false);
  const float2_t b = __builtin_amdgcn_cvt_pk_f32_fp8(x, true);
  return uint2{cvt_pk_bf16(a.x, a.y), cvt_pk_bf16(b.x, b.y)};
}

template <int HG, int SRC>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(Prefill a) {
  constexpr int RG = 4 / HG;                 // row groups of 32
  constexpr int TILE_ROWS = RG * WAVE_ROWS;
  constexpr int PARTS = SRC == ROWS ? 1 : 3;
  constexpr bool EACH = SRC == ROWS;         // rescale at each tile
  __shared__ __attribute__((aligned(16))) short lds[2][2][KV * HD];

  // Sequence s has the places seq_start[s] / TILE_ROWS + s and up, as many
  // as its tiles or more; the last places come first.
  const int w = gridDim.y - 1 - blockIdx.y;
  int s = 0;
  for (int hi = a.seqs; hi - s > 1;) {
    const int mid = (s + hi) >> 1;
    if (a.seq_start[mid] / TILE_ROWS + mid <= w) s = mid; else hi = mid;
  }
  const int t0 = a.seq_start[s], n = a.seq_start[s + 1] - t0;
  const int r0 = (w - t0 / TILE_ROWS - s) * TILE_ROWS;   // first row in s
  if (r0 >= n || n < a.min_rows) return;
  const int before = SRC == ROWS ? 0 : a.ctx_lens[t0] - 1;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, hf = lane >> 5;
  const int h = blockIdx.x * HG + wid % HG;
  const int g = blockIdx.x * HG / (a.H / a.G);   // one for HG heads
  const int rw = r0 + wid / HG * WAVE_ROWS;      // the wave's first row
  const int row = rw + col;
  const int last = before + min(r0 + TILE_ROWS, n) - 1;  // last token seen
  const int w_last = before + min(rw + WAVE_ROWS, n) - 1;

  short8_t qf[8];
  {
    const bf16* qp = a.q + (t0 + min(row, n - 1)) * a.sq + (long)h * HD;
    #pragma unroll
    for (int c = 0; c < 8; ++c)
      qf[c] = (*reinterpret_cast<const short8_t*>(qp + c * 16 + hf * 8) &
               a.q_and) ^ a.q_xor;
  }
  f32x16_t acc[4];
  #pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = f32x16_t(0.f);
  float m = -FLT_MAX, l = 0.f;

  // ---- tiles.  bf16: a wave brings 4 KB-units of K and of V, rows 16 j +
  // 4 wid and the three after it.  Tokens past the last one have a weight of
  // zero, which does not hide a NaN: beside q the last one is read again, in
  // the pages their values are cleared.  A tile's pages are looked up one tile
  // ahead.
  const int* bt = SRC == ROWS ? nullptr
                              : a.block_tables + (long)s * a.max_blocks;
  const int last_page = last / PAGE;
  int ids[4];
  auto look_up = [&](int kv0) {
    #pragma unroll
    for (int j = 0; j < 4; ++j)
      ids[j] = bt[min(kv0 / PAGE + j, last_page)];
  };
  const int lr = 4 * wid + (lane >> 4);          // row within 16
  const int kc = ((lane & 15) ^ lr) * 16;        // its byte of K, and of V
  const int vc = ((lane & 15) ^ (lane >> 4) << 2) * 16;
  uint4 raw[4];                                  // PAGES8: 32 bytes each
  auto fetch = [&](int kv0, int buf) {
    if constexpr (SRC == PAGES8) {
      const int tok = tid >> 2;
      const int id = ids[0] * (tok < 16) + ids[1] * (tok >> 4 == 1) +
                     ids[2] * (tok >> 4 == 2) + ids[3] * (tok >> 4 == 3);
      const long at = (((long)id * a.G + g) * PAGE + tok % PAGE) * HD +
                      (tid & 3) * 32;
      const char* kp = reinterpret_cast<const char*>(a.k) + at;
      const char* vp = reinterpret_cast<const char*>(a.v) + at;
      #pragma unroll
      for (int i = 0; i < 2; ++i) {
        raw[i] = reinterpret_cast<const uint4*>(kp)[i];
        raw[2 + i] = reinterpret_cast<const uint4*>(vp)[i];
      }
    } else {
      const RowLoads k_rows(a.k + (t0 + kv0) * a.sk + g * HD);
      const RowLoads v_rows(a.v + (t0 + kv0) * a.sv + g * HD);
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        char* kl = reinterpret_cast<char*>(
            &lds[buf][0][(16 * j + 4 * wid) * HD]);
        char* vl = reinterpret_cast<char*>(
            &lds[buf][1][(16 * j + 4 * wid) * HD]);
        if constexpr (SRC == ROWS) {
          const unsigned r = min(16 * j + lr, n - 1 - kv0);
          k_rows.to_lds(kl, r * (unsigned)a.sk * 2 + kc, 0);
          v_rows.to_lds(vl, r * (unsigned)a.sv * 2 + vc, 0);
        } else {
          const int id = __builtin_amdgcn_readfirstlane(ids[j]);
          const long at = ((long)id * a.G + g) * (PAGE * HD);
          RowLoads(a.k + at).to_lds(kl, lr * (HD * 2) + kc, 0);
          RowLoads(a.v + at).to_lds(vl, lr * (HD * 2) + vc, 0);
        }
      }
    }
  };
  auto store = [&](int kv0, int buf) {           // PAGES8
    const int tok = tid >> 2;
    if (kv0 + tok > last) raw[2] = raw[3] = uint4{0, 0, 0, 0};
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned* x = &raw[i].x;
      uint4 u[2];
      #pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint2 lo = widen(x[2 * j]), hi = widen(x[2 * j + 1]);
        u[j] = uint4{lo.x, lo.y, hi.x, hi.y};
      }
      #pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int c = (tid & 3) * 4 + (i & 1) * 2 + j;
        reinterpret_cast<uint4*>(lds[buf][i >> 1])
            [i < 2 ? k_unit(tok, c) : v_unit(tok, c)] = u[j];
      }
    }
  };

  // matrix row i of a 32-token block takes this token's key, so that
  // sc[b][r] is token 32 b + (r >> 3) * 16 + hf * 8 + (r & 7)
  const int krow = (col & 16) + ((col >> 2) & 1) * 8 + ((col >> 3) & 1) * 4 +
                   (col & 3);
  const int k_at = k_unit(krow, hf) * 16;        // bytes; step c: ^ c << 5
  // V^T: lane's part of a read of 4 tokens by 16 columns; block e: ^ e << 6
  const int vr = hf * 8 + ((lane & 15) >> 2);
  const int vcol = (lane >> 4 & 1) * 16 + (lane & 3) * 4;
  const int v_at = v_unit(vr, vcol >> 3) * 16 + (vcol & 7) * 2;

  auto compute = [&](int kv0, int buf) {
    const char* kl = reinterpret_cast<const char*>(lds[buf][0]);
    const char* vl = reinterpret_cast<const char*>(lds[buf][1]);
    f32x16_t sc[2];
    short8_t kf[8];
    auto key = [&](int b, int c) {
      return *reinterpret_cast<const short8_t*>(kl + (k_at ^ c << 5) +
                                                b * 32 * HD * 2);
    };
    #pragma unroll
    for (int c = 0; c < 8; ++c) kf[c] = key(0, c);
    sc[0] = sc[1] = f32x16_t(0.f);
    #pragma unroll
    for (int c = 0; c < 8; ++c) {
      sc[0] = mfma32(kf[c], qf[c], sc[0]);
      kf[c] = key(1, c);
    }
    #pragma unroll
    for (int c = 0; c < 8; ++c) sc[1] = mfma32(kf[c], qf[c], sc[1]);
    __builtin_amdgcn_sched_group_barrier(DS_READ, 8, 0);
    #pragma unroll
    for (int c = 0; c < 8; ++c) {
      __builtin_amdgcn_sched_group_barrier(PRODUCT, 1, 0);
      __builtin_amdgcn_sched_group_barrier(DS_READ, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(PRODUCT, 8, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (kv0 + KV - 1 > before + rw) {
      #pragma unroll
      for (int b = 0; b < 2; ++b)
        #pragma unroll
        for (int r = 0; r < 16; ++r)
          if (kv0 + b * 32 + (r >> 3) * 16 + hf * 8 + (r & 7) > before + row)
            sc[b][r] = -FLT_MAX;
    }
    float mx = -FLT_MAX;
    #pragma unroll
    for (int b = 0; b < 2; ++b)
      #pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[b][r]);
    mx = max_halves(mx) * a.scale;
    float alpha = 1.f;
    if (__any(mx > (EACH ? m : m + GROW))) {
      const float top = fmaxf(m, mx);
      alpha = m == -FLT_MAX ? 0.f
              : EACH ? __expf(m - top) : exp2_fast(m - top);
      #pragma unroll
      for (int e = 0; e < 4; ++e)
        #pragma unroll
        for (int r = 0; r < 16; ++r) acc[e][r] *= alpha;
      m = top;
    }
    const float base = m == -FLT_MAX ? 0.f : m;
    float sum = 0.f;
    union Values { short4_t h[2]; short8_t v; };
    Values vf[2][4];
    auto value = [&](int i, int e) {             // of tokens 16 i ..
      Values r;
      #pragma unroll
      for (int h = 0; h < 2; ++h)
        r.h[h] = lds_read_tr(reinterpret_cast<const short*>(
            vl + (v_at ^ e << 6) + (i * 16 + h * 4) * HD * 2));
      return r;
    };
    __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
    for (int e = 0; e < 4; ++e) vf[0][e] = value(0, e);
    short8_t part[2][PARTS];
    auto weigh = [&](int i, short8_t* to) {
      const int b = i >> 1, c = i & 1;
      float p[8];
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        p[j] = EACH ? __expf(product(sc[b][c * 8 + j], a.scale) - base)
                    : exp2_fast(fmaf(sc[b][c * 8 + j], a.scale, -base));
        if constexpr (!EACH) sum += p[j];
      }
      split_bf16x8<PARTS>(p, to);
      if constexpr (EACH) {
        // a lane sums 4 of every 8 tokens: t .. t + 3, t + 8 .. t + 11
        #pragma unroll
        for (int j = 0; j < 4; ++j) swap_halves(p[j], p[4 + j]);
        #pragma unroll
        for (int j = 0; j < 8; ++j) sum += p[j];
      }
    };
    weigh(0, part[0]);
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      if (i < 3) {
        #pragma unroll
        for (int e = 0; e < 4; ++e) vf[(i + 1) & 1][e] = value(i + 1, e);
        weigh(i + 1, part[(i + 1) & 1]);
      }
      #pragma unroll
      for (int e = 0; e < 4; ++e)
        #pragma unroll
        for (int n = 0; n < PARTS; ++n)
          acc[e] = mfma32(vf[i & 1][e].v, part[i & 1][n], acc[e]);
      // between the products the next values' loads and the next weights
      if (i < 3) {
        #pragma unroll
        for (int n = 0; n < 4 * PARTS; ++n) {
          __builtin_amdgcn_sched_group_barrier(PRODUCT, 1, 0);
          __builtin_amdgcn_sched_group_barrier(DS_READ, PARTS == 1 ? 2 : 1, 0);
          __builtin_amdgcn_sched_group_barrier(VALU, PARTS == 1 ? 12 : 6, 0);
        }
      }
    }
    if constexpr (EACH) {            // both halves, as the maximum
      float other = sum;
      swap_halves(sum, other);
      sum += other;
    }
    l = fmaf(l, alpha, sum);
  };

  auto landed = [&](int kv0, int buf) {
    if constexpr (SRC == PAGES8) store(kv0, buf);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (SRC == PAGES && kv0 + KV - 1 > last) {   // what this lane brought
      #pragma unroll
      for (int j = 0; j < 4; ++j)
        if (kv0 + 16 * j + lr > last)
          *reinterpret_cast<uint4*>(
              &lds[buf][1][(16 * j + 4 * wid) * HD + lane * 8]) =
              uint4{0, 0, 0, 0};
    }
    __syncthreads();
  };
  if constexpr (SRC != ROWS) look_up(0);
  fetch(0, 0);
  if constexpr (SRC != ROWS) look_up(KV);
  landed(0, 0);
  int buf = 0;
  for (int kv0 = 0; kv0 <= last; kv0 += KV, buf ^= 1) {
    const bool more = kv0 + KV <= last;
    if (more) {
      fetch(kv0 + KV, buf ^ 1);
      if constexpr (SRC != ROWS) look_up(kv0 + 2 * KV);
    }
    if (rw < n && kv0 <= w_last) compute(kv0, buf);
    if (more) landed(kv0 + KV, buf ^ 1);
  }

  if constexpr (!EACH) l += __shfl_xor(l, 32);
  if (row >= n) return;
  // acc[e][r]: column e * 32 + (r >> 2) * 8 + hf * 4 + (r & 3)
  const bool none = SRC == ROWS && !(l > 0.f);
  bf16* op = a.out + ((long)(t0 + row) * a.H + h) * HD + hf * 4;
  #pragma unroll
  for (int e = 0; e < 4; ++e)
    #pragma unroll
    for (int r = 0; r < 16; r += 4) {
      float x[4];
      #pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = none ? 0.f : acc[e][r + j] / l;
      *reinterpret_cast<uint2*>(op + e * 32 + r * 2) =
          uint2{cvt_pk_bf16(x[0], x[1]), cvt_pk_bf16(x[2], x[3])};
    }
}

template <int SRC>
void launch(const Prefill& p, long rows, hipStream_t stream) {
  if (rows == 0 || p.seqs == 0) return;
  Prefill a = p;
  a.q_and = a.scale == 0.f ? 0 : -1;
  a.q_xor = a.scale < 0.f ? (short)0x8000 : 0;
  a.scale = a.scale == 0.f ? 1.f : fabsf(a.scale);
  if (SRC != ROWS) a.scale *= LOG2E;
  const int group = a.H / a.G;
  #define RUN(HG)                                                           \
    attn_prefill_kernel<HG, SRC>                                            \
        <<<dim3((unsigned)(a.H / HG),                                       \
                (unsigned)(rows / (4 / HG * WAVE_ROWS) + a.seqs)),          \
           256, 0, stream>>>(a)
  if (group % 4 == 0) RUN(4);
  else if (group % 2 == 0) RUN(2);
  else RUN(1);
  #undef RUN
}

}  // namespace

void launch_attn_prefill_mfma(bf16* out, const bf16* q, const bf16* k,
                              const bf16* v, const int* seq_start,
                              int num_seqs, long rows, int num_heads,
                              int num_kv_heads, int head_dim, float scale,
                              long sq, long sk, long sv,
                              hipStream_t stream) {
  if (head_dim != HD)
    throw std::runtime_error("attn_prefill_mfma: head_dim must be 128");
  launch<ROWS>({out, q, k, v, seq_start, nullptr, nullptr, num_seqs,
                num_heads, num_kv_heads, 0, 0, scale, 0, 0, sq, sk, sv},
               rows, stream);
}

// portions of at least min_rows rows; the others' rows are left as they are
void launch_attn_prefill_paged(bf16* out, const bf16* q, const bf16* k_cache,
                               const bf16* v_cache, const int* block_tables,
                               const int* ctx_lens, const int* seq_start,
                               int num_seqs, long rows, int num_heads,
                               int num_kv_heads, int max_blocks, int min_rows,
                               float scale, long sq, bool kv_fp8,
                               hipStream_t stream) {
  const Prefill a{out, q, k_cache, v_cache, seq_start, ctx_lens, block_tables,
                  num_seqs, num_heads, num_kv_heads, max_blocks, min_rows,
                  scale, 0, 0, sq, 0, 0};
  if (kv_fp8)
    launch<PAGES8>(a, rows, stream);
  else
    launch<PAGES>(a, rows, stream);
}
