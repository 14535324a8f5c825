// Unified paged attention for gfx950 — serves the decode step (one query
// token per sequence), the rows of short portions, and prefill of other head
// sizes than 128 (attn_prefill_mfma.hip has that).
//
// Geometry of the general kernel (head_dim 64; wave64-native):
//   grid = (num_query_rows, num_kv_heads); block = 256 threads = 4 waves.
//   A workgroup owns one (row, kv_head): it processes the whole GQA group
//   (GROUP query heads) so K/V stream from HBM exactly once per group.
//   Waves split the KV pages round-robin (flash-decode style) with
//   per-head online-softmax state; a final LDS combine merges the waves.
//
//   K page read: 4 lanes per token x 64B slices -> 4 KiB coalesced/page.
//   V page read: lane owns a D/64-element column slice of all 16 rows.
//   v2 (profiles/r01: v1 was LDS-issue-bound at 155us/layer, 14x off
//   roofline): the lane's q slice lives in REGISTERS as raw bf16 pairs
//   (GROUP<=4) or is read as float4 from LDS (GROUP=8); score/softmax
//   LDS traffic is float4; V rows are preloaded per page.
//
// BLOCK_SIZE is fixed at 16 tokens (one KV page = 16 x 128 x 2B = 4 KiB
// per head — the pool unit sized for 288 GB HBM3E).
#include <float.h>

#include <type_traits>

#include "common.h"

#define ATTN_BS 16   // KV page size in tokens

template <int GROUP, int D>
__global__ __launch_bounds__(256) void paged_attn_kernel(
    bf16* __restrict__ out, const bf16* __restrict__ q,
    const bf16* __restrict__ k_cache, const bf16* __restrict__ v_cache,
    const int* __restrict__ block_tables, const int* __restrict__ ctx_lens,
    const int* __restrict__ row_seq, int max_blocks, int num_kv_heads,
    float scale, long q_stride) {
  constexpr int SLICE = D / 4;        // K elems per lane (4 lanes/token)
  constexpr int VPL = D / 64;         // V elems per lane (lane owns a slice)
  constexpr bool QREG = (GROUP <= 4); // q slice in registers vs LDS
  const int row = blockIdx.x;
  const int kvh = blockIdx.y;
  const int H = num_kv_heads * GROUP;
  const int ctx = ctx_lens[row];
  const int table = row_seq ? row_seq[row] : row;
  const int* bt = block_tables + (long)table * max_blocks;
  const int nblocks = (ctx + ATTN_BS - 1) / ATTN_BS;

  __shared__ __attribute__((aligned(16))) float q_lds[GROUP][D];
  __shared__ __attribute__((aligned(16))) float sc[4][GROUP][ATTN_BS];
  __shared__ __attribute__((aligned(16))) float comb_o[4][GROUP][D];
  __shared__ float comb_m[4][GROUP];
  __shared__ float comb_l[4][GROUP];

  const int wid = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int tok = lane >> 2;          // 0..15
  const int sl = lane & 3;            // K slice index
  const int d0 = sl * SLICE;

  // ---- stage the query group ----
  unsigned q_pk[QREG ? GROUP : 1][QREG ? SLICE / 2 : 1];  // raw bf16 pairs
  if constexpr (QREG) {
    const bf16* qp = q + (long)row * q_stride + (long)kvh * GROUP * D + d0;
    #pragma unroll
    for (int h = 0; h < GROUP; ++h) {
      #pragma unroll
      for (int i = 0; i < SLICE / 8; ++i) {
        uint4 r4 = *reinterpret_cast<const uint4*>(qp + h * D + i * 8);
        q_pk[h][i * 4 + 0] = r4.x;
        q_pk[h][i * 4 + 1] = r4.y;
        q_pk[h][i * 4 + 2] = r4.z;
        q_pk[h][i * 4 + 3] = r4.w;
      }
    }
  } else {
    for (int i = threadIdx.x; i < GROUP * D; i += 256) {
      const int h = i / D, d = i % D;
      q_lds[h][d] = bf2f(*(const unsigned short*)(
          q + (long)row * q_stride + (kvh * GROUP + h) * D + d));
    }
    __syncthreads();
  }

  float m[GROUP], l[GROUP], acc[GROUP][VPL];
  #pragma unroll
  for (int h = 0; h < GROUP; ++h) {
    m[h] = -FLT_MAX; l[h] = 0.f;
    #pragma unroll
    for (int i = 0; i < VPL; ++i) acc[h][i] = 0.f;
  }

  for (int b = wid; b < nblocks; b += 4) {
    const long blk = bt[b];
    const int nb = min(ATTN_BS, ctx - b * ATTN_BS);
    // ---- K dot: lane covers SLICE elems of its token's key ----
    unsigned k_pk[SLICE / 2];
    {
      const bf16* kp = k_cache +
          (((blk * num_kv_heads + kvh) * ATTN_BS + tok) * D + d0);
      #pragma unroll
      for (int i = 0; i < SLICE / 8; ++i) {
        uint4 r4 = *reinterpret_cast<const uint4*>(kp + i * 8);
        k_pk[i * 4 + 0] = r4.x;
        k_pk[i * 4 + 1] = r4.y;
        k_pk[i * 4 + 2] = r4.z;
        k_pk[i * 4 + 3] = r4.w;
      }
    }
    #pragma unroll
    for (int h = 0; h < GROUP; ++h) {
      float p = 0.f;
      if constexpr (QREG) {
        #pragma unroll
        for (int i = 0; i < SLICE / 2; ++i) {
          const unsigned qa = q_pk[h][i], ka = k_pk[i];
          p += bf2f((unsigned short)(qa & 0xffff)) *
               bf2f((unsigned short)(ka & 0xffff));
          p += bf2f((unsigned short)(qa >> 16)) *
               bf2f((unsigned short)(ka >> 16));
        }
      } else {
        #pragma unroll
        for (int i = 0; i < SLICE / 4; ++i) {
          const float4 qv = *reinterpret_cast<const float4*>(
              &q_lds[h][d0 + i * 4]);
          p += qv.x * bf2f((unsigned short)(k_pk[i * 2] & 0xffff));
          p += qv.y * bf2f((unsigned short)(k_pk[i * 2] >> 16));
          p += qv.z * bf2f((unsigned short)(k_pk[i * 2 + 1] & 0xffff));
          p += qv.w * bf2f((unsigned short)(k_pk[i * 2 + 1] >> 16));
        }
      }
      p += __shfl_xor(p, 1);
      p += __shfl_xor(p, 2);
      if (sl == 0)
        sc[wid][h][tok] = (tok < nb) ? p * scale : -FLT_MAX;
    }
    // wave-private LDS area; DS ops of one wave are in program order.
    // ---- online softmax update + exponentiate in LDS ----
    float mn_h[GROUP];
    #pragma unroll
    for (int h = 0; h < GROUP; ++h) {
      float bm = -FLT_MAX;
      #pragma unroll
      for (int t4 = 0; t4 < ATTN_BS / 4; ++t4) {
        const float4 s4 = *reinterpret_cast<const float4*>(
            &sc[wid][h][t4 * 4]);
        bm = fmaxf(fmaxf(bm, fmaxf(s4.x, s4.y)), fmaxf(s4.z, s4.w));
      }
      const float mn = fmaxf(m[h], bm);
      mn_h[h] = mn;
      const float alpha = (m[h] == -FLT_MAX) ? 0.f : __expf(m[h] - mn);
      #pragma unroll
      for (int i = 0; i < VPL; ++i) acc[h][i] *= alpha;
      l[h] *= alpha;
      m[h] = mn;
      if (sl == 0)  // one lane per token exponentiates it
        sc[wid][h][tok] = (tok < nb) ? __expf(sc[wid][h][tok] - mn) : 0.f;
    }
    // ---- V: preload the lane's column slice of all 16 rows ----
    const bf16* vbase = v_cache +
        ((blk * num_kv_heads + kvh) * ATTN_BS) * D + lane * VPL;
    float vf[ATTN_BS][VPL];
    #pragma unroll
    for (int t = 0; t < ATTN_BS; ++t) {
      if (t < nb) {
        if constexpr (VPL == 2) {
          ushort2 vv = *reinterpret_cast<const ushort2*>(vbase + (long)t * D);
          vf[t][0] = bf2f(vv.x); vf[t][1] = bf2f(vv.y);
        } else {
          vf[t][0] = bf2f(*(const unsigned short*)(vbase + (long)t * D));
        }
      } else {
        #pragma unroll
        for (int i = 0; i < VPL; ++i) vf[t][i] = 0.f;
      }
    }
    #pragma unroll
    for (int h = 0; h < GROUP; ++h) {
      float s = 0.f;
      #pragma unroll
      for (int t4 = 0; t4 < ATTN_BS / 4; ++t4) {
        const float4 p4 = *reinterpret_cast<const float4*>(
            &sc[wid][h][t4 * 4]);
        #pragma unroll
        for (int i = 0; i < VPL; ++i) {
          acc[h][i] += p4.x * vf[t4 * 4 + 0][i];
          acc[h][i] += p4.y * vf[t4 * 4 + 1][i];
          acc[h][i] += p4.z * vf[t4 * 4 + 2][i];
          acc[h][i] += p4.w * vf[t4 * 4 + 3][i];
        }
        s += p4.x + p4.y + p4.z + p4.w;
      }
      l[h] += s;
      (void)mn_h;
    }
  }

  // ---- combine the 4 waves ----
  #pragma unroll
  for (int h = 0; h < GROUP; ++h) {
    #pragma unroll
    for (int i = 0; i < VPL; ++i) comb_o[wid][h][lane * VPL + i] = acc[h][i];
    if (lane == 0) { comb_m[wid][h] = m[h]; comb_l[wid][h] = l[h]; }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < GROUP * D; i += 256) {
    const int h = i / D, d = i % D;
    float M = fmaxf(fmaxf(comb_m[0][h], comb_m[1][h]),
                    fmaxf(comb_m[2][h], comb_m[3][h]));
    float o = 0.f, L = 0.f;
    #pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = (comb_m[w][h] == -FLT_MAX) ? 0.f
                                                 : __expf(comb_m[w][h] - M);
      o += f * comb_o[w][h][d];
      L += f * comb_l[w][h];
    }
    *(unsigned short*)(out + ((long)row * H + kvh * GROUP + h) * D + d) =
        f2bf(o / L);
  }
}

// ---------------------------------------------------------------------------
// head_dim 128: matrix cores (v_mfma_f32_16x16x32_bf16).
//
// What bounds it: reading the pages once, about 6 TB/s.  A dot product of four
// heads with a token on the vector units takes longer than the token's 512
// bytes; so up to 16 heads of a kv head are the columns of a product, however
// few they are.  Scores are formed transposed, S^T = K Q^T, with the K row
// that feeds matrix row i permuted so that the scores a lane holds are 8
// consecutive tokens of one head, the operand P^T of O^T = V^T P^T; the
// weights, floats, enter as three bf16 parts.  K goes from memory to its
// operands; V is turned by an LDS tile of the wave's own and the transposing
// LDS load, e4m3 pages are widened on the way.  A wave has 32 tokens at a time
// and issues the next ones' loads as soon as these are in their operands; no
// barrier until the waves' parts are added up.  Decoded rows read pages of their own
// once, by non-temporal loads, which do not wait for a place in the unit's cache: a
// step of 8 layers of 256 rows of about 1000 tokens 3019 -> 2903 us, of 8 of 8000 1249
// -> 1237, of 32 with 4 kv heads 548 -> 537, 1 of 1000 839 -> 833.  Such a load has
// whole lines: of K 128 bytes of 8 rows, and two exchange halves across lanes (64 of
// 16 rows, the operands, asked for every line twice): 32 x 4 kv heads of 1000 21.1 ->
// 19.8 us, 256 x 8 188 -> 182, e4m3 64 x 8 32.2 -> 30.9, but 8 of 8000 in two parts
// 50.2 50.9; the steps 2918 -> 2888, 1222 -> 1198 and 533 -> 524.
//
// Rows that begin with the same prompt share its pages, and pages that others read
// too are slower so.  They are looked for where one of the next 16 rows begins with
// the same page: its table is read along, and what both name is loaded as usual.  us
// with all pages by non-temporal loads, none, and so, 100 tokens of each row's own: 32
// x 4 kv heads after 1024 shared tokens 17.7 14.7 15.4, 16 x 8 after 8192 75.7 52.6
// 54.0, 256 x 8 in 8 groups after 4096 each 475 322 320; with 1000 of their own 256 x
// 8 after 1024 222 228 216; without shared pages 256 x 8 of 1000 170 188 168, 32 x 4
// 17.9 19.9 18.1, 8 of 8000 47.0 53.6 47.4.  Steps of 8 layers, all non-temporal and
// so: 32 narrow rows after 1024 shared tokens 502 -> 481, 16 after 8192 1306 -> 1234, 64
// after 2048 1311 -> 1293, 256 after 512 2344 -> 2331.
//
// us against dot products on the vector units, ragged contexts around the
// mean: 256 rows x 8 kv heads of 4, 1000 tokens 239 -> 208 (5.0 TB/s), with
// e4m3 pages 214 -> 110; 64 rows 77 -> 59, e4m3 71 -> 32; 8 rows of 8000 in 4
// parts 122 -> 61; 64 rows x 1 kv head of 8 in 4 parts 47 -> 16.
//
// ROPE: q and k come as the projection left them.  A lane turns its part of q
// in its registers; the wave that has the row's last token turns k and stores
// it and v before it loads the last block.  A launch of its own for that is one
// workgroup a token that goes to memory three times in a row, 5 us a layer;
// here these loads pass beside the page ids and the first pages.  us of both
// launches and of one: 1 row x 8 kv heads of 4, 1000 tokens 12.6 -> 10.1; 8
// rows of 8000 69 -> 63; 32 x 4 of 1000 27.7 -> 23.6; 256 x 8 of 1000 221 ->
// 206, of 30 22.4 -> 21.9; e4m3 64 x 8 of 1000 38.5 -> 34.8.
//
// SPLIT > 1 (flash-decode): `split` workgroups share one (row, kvh), each
// with every split-th 4 blocks of 32 tokens; their (o, m, l) land in
// `partial` [rows, kvh, split, group, D + 2] and a second kernel merges them.
// ---------------------------------------------------------------------------
namespace {

constexpr int HD = 128;
constexpr int BLOCK = 32;            // tokens a wave has at a time
constexpr float LOG2E = 1.4426950408889634f;
constexpr float GROW = 8.f;          // rescale when a maximum grows by 2^GROW

typedef __attribute__((ext_vector_type(4))) short short4_t;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(2))) float float2_t;

DEV float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// four rows of one column: in every 16 lanes, lane i passes the address of
// row i / 4, columns 4 (i % 4), and receives column i
DEV short4_t lds_read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) short4_t*)p);
}

// byte of 16-byte unit c of row r of a V tile: what 32 lanes read at a time,
// 64 bytes of rows r .. r + 3 and r + 8 .. r + 11, has a bank each
DEV int v_byte(int r, int c) {
  return r * 256 + ((c ^ (r & 3) << 2 ^ (r >> 3 & 1) << 1) << 4);
}

// 4 e4m3 bytes as bf16, exactly
DEV uint2 widen(unsigned x) {
  const float2_t a = __builtin_amdgcn_cvt_pk_f32_fp8(x, false);
  const float2_t b = __builtin_amdgcn_cvt_pk_f32_fp8(x, true);
  return uint2{cvt_pk_bf16(a.x, a.y), cvt_pk_bf16(b.x, b.y)};
}
DEV u32x4 widen(unsigned x, unsigned y) {
  const uint2 a = widen(x), b = widen(y);
  return u32x4{a.x, a.y, b.x, b.y};
}

// (x, y) by an angle, rounded as in rope_kv_append
DEV float2 turn(float x, float y, float c, float s) {
  return make_float2(fmaf(x, c, -(y * s)), fmaf(y, c, x * s));
}

struct Paged {
  bf16* out;
  const bf16* q;
  const void* k_cache;
  const void* v_cache;
  const int* block_tables;
  const int* ctx_lens;
  const int* row_seq;
  const int* seq_start;      // with row_seq: only sequences of at most
  int max_portion;           // max_portion rows
  int max_blocks, G, group;
  float scale;               // times log2(e)
  long qs;
  float* partial;
  // ROPE: rows are the last tokens of different sequences
  const bf16* k;
  const bf16* v;
  const float* cos_sin;      // [positions, HD], cosines | sines
  const long* positions;
  const long* slots;         // -1: nothing is stored
  long ks, vs;
  int rows, split;
};

constexpr unsigned GRID_Y = 65535;
constexpr int NEAR = 16;             // rows after a row that are looked at

template <bool KV8, bool ROPE>
__global__ __launch_bounds__(256, 3) void paged_attn_mfma_kernel(Paged a) {
  __shared__ __attribute__((aligned(16))) char v_lds[4][BLOCK * HD * 2];
  __shared__ float m_lds[4][16], l_lds[4][16];
  // Without parts the heads of a row, whose pages lie beside each other, come
  // first, which memory reads faster than rows first where contexts are ragged:
  // us of a step of 8 layers with 8 kv heads of 4, 256 rows of about 1000 tokens
  // 3236 -> 3102, of 64 1775 1765, 100 of 1000 1908 -> 1859; of 4 layers with e4m3
  // pages, 256 of 1000 1120 -> 1059, of 64 741 -> 707; 8 layers with 4 kv heads 256
  // of 1000 1577 1564; within 1 % with 64 rows.  Contexts of one length read as
  // fast either way (the attention alone 196 194), and 64 tokens of each slower
  // (19.6 20.3, e4m3 15.0 16.3).  With parts, rows first (8 x 8 of 8000 in 4 parts
  // 54, the other way 55).
  const int group = a.group, split = a.split;
  const bool whole = split == 1;
  const int g = whole ? blockIdx.x : blockIdx.y;
  const int row = whole ? blockIdx.y + blockIdx.z * GRID_Y : blockIdx.x;
  const int z = whole ? 0 : blockIdx.z;
  if (row >= a.rows) return;
  const int table = a.row_seq ? a.row_seq[row] : row;
  if (a.seq_start &&
      a.seq_start[table + 1] - a.seq_start[table] > a.max_portion)
    return;
  const int ctx = a.ctx_lens[row];
  const int lane = threadIdx.x & 63;
  // ROPE: where the next rows begin, and how long they are
  int near_page = 0, near_ctx = 0, near_row = row;
  if constexpr (ROPE) {
    near_row += 1 + lane % NEAR;
    if (near_row >= a.rows) near_row -= a.rows;
    if (near_row >= a.rows) near_row = row;
    near_page = a.block_tables[(long)near_row * a.max_blocks];
    near_ctx = a.ctx_lens[near_row];
  }
  // scalar loads also after the stores to the pages
  typedef const __attribute__((address_space(4))) int* Ints;
  const auto bt = (Ints)(a.block_tables + (long)table * a.max_blocks);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, gr = lane >> 4;

  // step c of the score product has columns 32 c + 8 gr; with e4m3, of which
  // a lane reads 16 at a time, 64 (c / 2) + 16 gr + 8 (c % 2)
  short8_t qf[4];
  #pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int d = KV8 ? (c >> 1) * 64 + gr * 16 + (c & 1) * 8
                      : c * 32 + gr * 8;
    qf[c] = col < group
        ? *reinterpret_cast<const short8_t*>(
              a.q + row * a.qs + (long)(g * group + col) * HD + d)
        : short8_t{};
  }
  constexpr int ELEM = KV8 ? 1 : 2;
  // to turn with, loaded before the first pages: of steps c and c + 2, columns
  // d and d + 64; and by the wave that has the row's last token
  f32x4_t co[2][2], si[2][2];
  bool append = false;
  float2 co_k, si_k;                 // lanes 0 to 31: columns j, j + 1 of k
  unsigned lo = 0, hi = 0;           // and j + 64, j + 65; the others: 4 of v
  long slot = -1;
  const int j_new = lane % 32 * 2;
  if constexpr (ROPE) {
    const float* cs = a.cos_sin + a.positions[row] * HD;
    slot = a.slots[row];
    append = slot >= 0 &&
             max(ctx - 1, 0) / BLOCK % (4 * split) == z * 4 + wid;
    #pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int d = KV8 ? gr * 16 + c * 8 : c * 32 + gr * 8;
      #pragma unroll
      for (int i = 0; i < 2; ++i) {
        co[c][i] = *reinterpret_cast<const f32x4_t*>(cs + d + i * 4);
        si[c][i] = *reinterpret_cast<const f32x4_t*>(cs + HD / 2 + d + i * 4);
      }
    }
    if (append) {
      co_k = *reinterpret_cast<const float2*>(cs + j_new);
      si_k = *reinterpret_cast<const float2*>(cs + HD / 2 + j_new);
      const bf16* p = lane < 32 ? a.k + row * a.ks + g * HD + j_new
                                : a.v + row * a.vs + g * HD + j_new * 2;
      lo = *reinterpret_cast<const unsigned*>(p);
      hi = *reinterpret_cast<const unsigned*>(p + (lane < 32 ? HD / 2 : 2));
    }
  }
  f32x4_t acc[8];
  #pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = f32x4_t(0.f);
  float m = -FLT_MAX, l = 0.f;

  // matrix row i of half t takes token 8 (i / 4) + 4 t + i % 4
  // of a page: rows 0 to 7 are on the first, 8 to 15 on the second; a load has the
  // whole lines of 8 rows, and two exchange halves
  const int k_at = (8 * (col >> 2 & 1) + (col & 3)) * (HD * ELEM) +
                   (col >> 3) * 64 + gr * 16;
  const int blocks = (ctx + BLOCK - 1) / BLOCK;
  const int last_page = (ctx - 1) / ATTN_BS;
  const int step = 4 * split;
  long b0 = 0, b1 = 0;               // page ids, read one block ahead
  auto bn = bt;                      // a row that begins as this one,
  int n0 = 0, shared = 0;            // its page there, and its blocks
  bool both = false;
  if constexpr (ROPE) {              // known with the first page: the next row
    const int next = row + 1 < a.rows ? row + 1 : 0;
    bn = (Ints)(a.block_tables + (long)next * a.max_blocks);
    const int of = ((Ints)a.ctx_lens)[next];
    if (next != row && bn[0] == bt[0]) shared = of / BLOCK;
  }
  auto pages = [&](int i) {
    b0 = bt[min(2 * i, last_page)];
    b1 = bt[min(2 * i + 1, last_page)];
    n0 = bn[min(2 * i, last_page)];
    both = i < shared;
  };
  u32x4 kr[2][KV8 ? 2 : 4], vr[KV8 ? 4 : 8];
  auto load = [&](auto once) {
    auto page = [](const char* p) {
      const auto at = reinterpret_cast<const u32x4*>(p);
      return decltype(once)::value ? __builtin_nontemporal_load(at) : *at;
    };
    const long p0 = (b0 * a.G + g) * (ATTN_BS * HD * ELEM);
    const long p1 = (b1 * a.G + g) * (ATTN_BS * HD * ELEM);
    const char* kc = static_cast<const char*>(a.k_cache);
    const char* vc = static_cast<const char*>(a.v_cache);
    #pragma unroll
    for (int t = 0; t < 2; ++t)
      #pragma unroll
      for (int c = 0; c < (KV8 ? 2 : 4); ++c)
        kr[t][c] = page(kc + (c & 1 ? p1 : p0) + k_at + 4 * t * HD * ELEM +
                        (c >> 1) * 128);
    #pragma unroll
    for (int i = 0; i < (KV8 ? 4 : 8); ++i)
      vr[i] = page(vc + (i < (KV8 ? 2 : 4) ? p0 : p1) +
                   (i % (KV8 ? 2 : 4)) * 1024 + lane * 16);
  };
  // Rows of a portion share its pages.  The two ways differ by more than the hint,
  // or the compiler makes one of them, without it.
  auto fetch = [&]() {
    if (!ROPE || (both && n0 == (int)b0)) {
      load(std::false_type());
    } else {
      asm volatile("; read once" ::: "memory");
      load(std::true_type());
      asm volatile("; read once" ::: "memory");
    }
  };
  char* vl = v_lds[wid];
  const int vr0 = gr * 8 + (col >> 2);
  const int v_at = v_byte(vr0, (col & 3) >> 1) + (col & 1) * 8;

  int i = z * 4 + wid;
  const bool at_once = !append || i + step < blocks;   // else stored first
  if (i < blocks) {
    pages(i);
    if (at_once) {
      fetch();
      if (ROPE && !shared) {         // others, not waited for until here
        const auto with = __ballot(near_page == bt[0] && near_row != row &&
                                   near_ctx >= 2 * BLOCK);
        if (with) {
          const int l = __ffsll(with) - 1;
          bn = (Ints)(a.block_tables +
                      (long)__builtin_amdgcn_readlane(near_row, l) *
                          a.max_blocks);
          shared = __builtin_amdgcn_readlane(near_ctx, l) / BLOCK;
        }
      }
      if (i + step < blocks) pages(i + step);
    }
  }
  if constexpr (ROPE) {
    #pragma unroll
    for (int c = 0; c < 2; ++c)
      #pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = bf2f((unsigned short)qf[c][i]);
        const float y = bf2f((unsigned short)qf[c + 2][i]);
        const float2 r = turn(x, y, co[c][i >> 2][i & 3],
                              si[c][i >> 2][i & 3]);
        qf[c][i] = (short)f2bf(r.x);
        qf[c + 2][i] = (short)f2bf(r.y);
      }
    if (append) {
      const long at =
          ((slot / ATTN_BS * a.G + g) * ATTN_BS + slot % ATTN_BS) * HD * ELEM;
      char* kp = static_cast<char*>(const_cast<void*>(a.k_cache)) + at;
      char* vp = static_cast<char*>(const_cast<void*>(a.v_cache)) + at;
      const int j = j_new;
      const float x0 = __uint_as_float(lo << 16);
      const float x1 = __uint_as_float(lo & 0xffff0000u);
      const float y0 = __uint_as_float(hi << 16);
      const float y1 = __uint_as_float(hi & 0xffff0000u);
      if (lane < 32) {
        const float2 t0 = turn(x0, y0, co_k.x, si_k.x);
        const float2 t1 = turn(x1, y1, co_k.y, si_k.y);
        if constexpr (KV8) {
          *reinterpret_cast<unsigned short*>(kp + j) = (unsigned short)
              __builtin_amdgcn_cvt_pk_fp8_f32(t0.x, t1.x, 0, false);
          *reinterpret_cast<unsigned short*>(kp + HD / 2 + j) =
              (unsigned short)__builtin_amdgcn_cvt_pk_fp8_f32(t0.y, t1.y, 0,
                                                              false);
        } else {
          *reinterpret_cast<unsigned*>(kp + j * 2) = cvt_pk_bf16(t0.x, t1.x);
          *reinterpret_cast<unsigned*>(kp + HD + j * 2) =
              cvt_pk_bf16(t0.y, t1.y);
        }
      } else if constexpr (KV8) {
        const int w = __builtin_amdgcn_cvt_pk_fp8_f32(x0, x1, 0, false);
        *reinterpret_cast<int*>(vp + j * 2) =
            __builtin_amdgcn_cvt_pk_fp8_f32(y0, y1, w, true);
      } else {
        *reinterpret_cast<uint2*>(vp + j * 4) = uint2{lo, hi};
      }
      if (!at_once && i < blocks) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        load(std::true_type());
      }
    }
  }
  for (; i < blocks; i += step) {
    f32x4_t sc[2];
    #pragma unroll
    for (int t = 0; t < 2; ++t) {
      #pragma unroll
      for (int c = 0; c < (KV8 ? 2 : 4); c += 2)
        exchange_halves(kr[t][c], kr[t][c + 1]);
      sc[t] = f32x4_t(0.f);
      #pragma unroll
      for (int c = 0; c < 4; ++c) {
        union { u32x4 u; short8_t v; } k;
        if constexpr (KV8) {
          const u32x4 x = kr[t][c >> 1];
          k.u = c & 1 ? widen(x.z, x.w) : widen(x.x, x.y);
        } else {
          k.u = kr[t][c];
        }
        sc[t] = mfma16(k.v, qf[c], sc[t]);
      }
    }
    // what the page holds after the last token: a weight of zero does not hide
    // a NaN
    if ((i + 1) * BLOCK > ctx) {
      #pragma unroll
      for (int j = 0; j < (KV8 ? 4 : 8); ++j)
        if (i * BLOCK + (KV8 ? 8 * j + (lane >> 3) : 4 * j + gr) >= ctx)
          vr[j] = u32x4(0);
    }
    if constexpr (KV8) {             // rows 8 j + lane / 8
      #pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = 8 * j + (lane >> 3), c = (lane & 7) * 2;
        *reinterpret_cast<u32x4*>(vl + v_byte(r, c)) =
            widen(vr[j].x, vr[j].y);
        *reinterpret_cast<u32x4*>(vl + v_byte(r, c + 1)) =
            widen(vr[j].z, vr[j].w);
      }
    } else {                         // rows 4 j + lane / 16
      #pragma unroll
      for (int j = 0; j < 8; ++j)
        *reinterpret_cast<u32x4*>(vl + v_byte(4 * j + gr, col)) = vr[j];
    }
    if (i + step < blocks) {
      // before the wave's last block: what it stored is in the page
      if (ROPE && append && i + 2 * step >= blocks)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
      fetch();
      if (i + 2 * step < blocks) pages(i + 2 * step);
    }
    float p[8], mx = -FLT_MAX;
    #pragma unroll
    for (int j = 0; j < 8; ++j) p[j] = sc[j >> 2][j & 3] * a.scale;
    if ((i + 1) * BLOCK > ctx) {
      #pragma unroll
      for (int j = 0; j < 8; ++j)
        if (i * BLOCK + gr * 8 + j >= ctx) p[j] = -FLT_MAX;
    }
    #pragma unroll
    for (int j = 0; j < 8; ++j) mx = fmaxf(mx, p[j]);
    mx = reduce_32(reduce_16(mx, MaxOf()), MaxOf());
    if (__any(mx > m + GROW)) {
      const float top = fmaxf(m, mx);
      const float alpha = m == -FLT_MAX ? 0.f : exp2_fast(m - top);
      #pragma unroll
      for (int e = 0; e < 8; ++e)
        #pragma unroll
        for (int r = 0; r < 4; ++r) acc[e][r] *= alpha;
      l *= alpha;
      m = top;
    }
    const float base = m == -FLT_MAX ? 0.f : m;
    #pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = exp2_fast(p[j] - base);
      l += p[j];
    }
    short8_t part[3];
    split_bf16x8<3>(p, part);
    #pragma unroll
    for (int e = 0; e < 8; ++e) {
      union { short4_t h[2]; short8_t v; } vf;
      // row + 4: the same units; column block e: two units on
      vf.h[0] = lds_read_tr(vl + (v_at ^ e << 5));
      vf.h[1] = lds_read_tr(vl + (v_at ^ e << 5) + 4 * 256);
      #pragma unroll
      for (int n = 0; n < 3; ++n) acc[e] = mfma16(vf.v, part[n], acc[e]);
    }
  }
  l = reduce_32(reduce_16(l, SumOf()), SumOf());
  __syncthreads();
  float* comb = reinterpret_cast<float*>(v_lds);     // [4][group][HD]
  if (gr == 0) {
    m_lds[wid][col] = m;
    l_lds[wid][col] = l;
  }
  if (col < group) {
    #pragma unroll
    for (int e = 0; e < 8; ++e)
      *reinterpret_cast<f32x4_t*>(
          comb + (wid * group + col) * HD + e * 16 + gr * 4) = acc[e];
  }
  __syncthreads();
  for (int u = threadIdx.x * 4; u < group * HD; u += 1024) {
    const int h = u / HD, d = u % HD;
    float top = -FLT_MAX, sum = 0.f;
    #pragma unroll
    for (int w = 0; w < 4; ++w) top = fmaxf(top, m_lds[w][h]);
    f32x4_t o = f32x4_t(0.f);
    #pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = m_lds[w][h];
      const float f = mw == -FLT_MAX ? 0.f : exp2_fast(mw - top);
      sum += f * l_lds[w][h];
      o += *reinterpret_cast<const f32x4_t*>(comb + w * group * HD + u) * f;
    }
    if (split == 1) {
      const float inv = 1.f / sum;
      *reinterpret_cast<uint2*>(
          a.out + (((long)row * a.G + g) * group + h) * HD + d) =
          uint2{cvt_pk_bf16(o[0] * inv, o[1] * inv),
                cvt_pk_bf16(o[2] * inv, o[3] * inv)};
    } else {
      float* pr = a.partial +
          ((((long)row * a.G + g) * split + z) * group + h) * (HD + 2);
      // rows of 130 floats: 8-byte aligned
      *reinterpret_cast<float2*>(pr + d) = make_float2(o[0], o[1]);
      *reinterpret_cast<float2*>(pr + d + 2) = make_float2(o[2], o[3]);
      if (d == 0) *reinterpret_cast<float2*>(pr + HD) = make_float2(top, sum);
    }
  }
}

// The parts of one (row, head) a wave, two columns a lane; lane z has part z's
// maximum and sum, so that all loads are independent, and those of 16 parts are
// issued before the first is needed (one workgroup a (row, kvh) that walked the
// parts took 17 us for one row, 16 parts; 4 rows in 8 parts, attention over 32
// tokens included, 8.0 us with the loads after the sums, 6.8 so).
__global__ __launch_bounds__(256) void paged_attn_merge_kernel(
    bf16* __restrict__ out, const float* __restrict__ partial, int split,
    int group, long heads) {
  const long rh = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (rh >= heads) return;
  const int lane = threadIdx.x & 63, h = (int)(rh % group);
  const float* base = partial + (rh / group * split * group + h) * (HD + 2);
  const long stride = (long)group * (HD + 2);
  float2 o[16];                      // also the first parts' columns
  auto load = [&](int z0) {
    #pragma unroll
    for (int z = 0; z < 16; ++z)
      if (z0 + z < split)
        o[z] = *reinterpret_cast<const float2*>(
            base + (z0 + z) * stride + lane * 2);
  };
  float2 ml = make_float2(-FLT_MAX, 0.f);
  if (lane < split)
    ml = *reinterpret_cast<const float2*>(base + lane * stride + HD);
  load(0);
  const float top = wave_reduce_max(ml.x);
  const float f = ml.x == -FLT_MAX ? 0.f : exp2_fast(ml.x - top);
  const float sum = wave_reduce_sum(f * ml.y);
  float x = 0.f, y = 0.f;
  for (int z0 = 0;;) {
    #pragma unroll
    for (int z = 0; z < 16; ++z)
      if (z0 + z < split) {
        const float fz = __shfl(f, z0 + z);
        x += fz * o[z].x;
        y += fz * o[z].y;
      }
    if ((z0 += 16) >= split) break;
    load(z0);
  }
  const float inv = 1.f / sum;
  *reinterpret_cast<unsigned*>(out + rh * HD + lane * 2) =
      cvt_pk_bf16(x * inv, y * inv);
}

template <bool ROPE>
void launch_mfma(Paged a, long rows, int split, bool kv_fp8,
                 hipStream_t stream) {
  a.rows = (int)rows;
  a.split = split;
  const unsigned n = (unsigned)rows;
  const dim3 grid = split == 1
      ? dim3((unsigned)a.G, n < GRID_Y ? n : GRID_Y, (n + GRID_Y - 1) / GRID_Y)
      : dim3(n, (unsigned)a.G, (unsigned)split);
  if (kv_fp8)
    paged_attn_mfma_kernel<true, ROPE><<<grid, 256, 0, stream>>>(a);
  else
    paged_attn_mfma_kernel<false, ROPE><<<grid, 256, 0, stream>>>(a);
  if (split > 1) {
    const long heads = rows * a.G * a.group;
    paged_attn_merge_kernel<<<(unsigned)((heads + 3) / 4), 256, 0, stream>>>(
        a.out, a.partial, split, a.group, heads);
  }
}

}  // namespace

// With seq_start (and row_seq) only the rows of sequences that have at most
// max_portion rows are computed.
void launch_paged_attn(bf16* out, const bf16* q, const bf16* k_cache,
                       const bf16* v_cache, const int* block_tables,
                       const int* ctx_lens, const int* row_seq,
                       long num_rows, int num_kv_heads, int group, int D,
                       int max_blocks, int block_size, float scale,
                       long q_stride, float* split_ws, int split,
                       bool kv_fp8, const int* seq_start, int max_portion,
                       hipStream_t stream) {
  if (block_size != ATTN_BS)
    throw std::runtime_error("paged_attn: block_size must be 16");
  if (D == HD && (group <= 4 || group == 8)) {
    if (split > 64)
      throw std::runtime_error("paged_attn: at most 64 parts");
    launch_mfma<false>({out, q, k_cache, v_cache, block_tables, ctx_lens,
                        row_seq, seq_start, max_portion, max_blocks,
                        num_kv_heads, group, scale * LOG2E, q_stride,
                        split_ws}, num_rows, split, kv_fp8, stream);
    return;
  }
  if (split != 1 || seq_start)
    throw std::runtime_error("paged_attn: split needs head_dim 128");
  if (kv_fp8)
    throw std::runtime_error("paged_attn: fp8 KV needs head_dim 128");
  dim3 grid((unsigned)num_rows, (unsigned)num_kv_heads);
  #define CASE(G, DD)                                                       \
    if (group == G && D == DD) {                                            \
      paged_attn_kernel<G, DD><<<grid, 256, 0, stream>>>(                   \
          out, q, k_cache, v_cache, block_tables, ctx_lens, row_seq,        \
          max_blocks, num_kv_heads, scale, q_stride);                       \
      return;                                                               \
    }
  CASE(1, 64) CASE(2, 64) CASE(4, 64) CASE(8, 64)
  #undef CASE
  throw std::runtime_error("paged_attn: unsupported (group, head_dim)");
}

// rope_kv_append and paged_attn of one token each of different sequences: q
// [rows, kv heads * group, 128] as they come from the projection, rows 16-byte
// aligned; q and k stay as they are.
void launch_rope_paged_attn(bf16* out, const bf16* q, const bf16* k,
                            const bf16* v, const long* positions,
                            const float* cos_sin, const long* slots,
                            bf16* k_cache, bf16* v_cache,
                            const int* block_tables, const int* ctx_lens,
                            long rows, int num_kv_heads, int group,
                            int max_blocks, float scale, long qs, long ks,
                            long vs, float* split_ws, int split, bool kv_fp8,
                            hipStream_t stream) {
  // every row's first page is read, also where no row has a page
  if (max_blocks == 0) block_tables = ctx_lens;
  launch_mfma<true>({out, q, k_cache, v_cache, block_tables, ctx_lens, nullptr,
                     nullptr, 0, max_blocks, num_kv_heads, group,
                     scale * LOG2E, qs, split_ws, k, v, cos_sin, positions,
                     slots, ks, vs}, rows, split, kv_fp8, stream);
}
