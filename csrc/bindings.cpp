// Python bindings for the gfx950 kernel set (hyperspot._C).
//
// Host-side glue only — every kernel lives in a .hip translation unit and
// is reached through a plain launcher so this file needs no device code.
#include "bindings.h"

#include <array>

#include "recurrent.h"

void launch_rmsnorm(bf16*, const bf16*, const bf16*, float, long, int,
                    hipStream_t);
void launch_parts_add_rmsnorm(bf16*, const float*, int, bf16*, const bf16*,
                              float, long, int, hipStream_t);
void launch_choices_add_rmsnorm(bf16*, const bf16*, const int*, const float*,
                                int, bf16*, const bf16*, float, long, int,
                                hipStream_t);
void launch_fused_add_rmsnorm(bf16*, bf16*, const bf16*, float, long, int,
                              hipStream_t);
void launch_rope_kv_append(bf16*, bf16*, const bf16*, const long*,
                           const float*, const long*, bf16*, bf16*, long,
                           int, int, int, int, long, long, long, bool,
                           hipStream_t);
void launch_paged_attn(bf16*, const bf16*, const bf16*, const bf16*,
                       const int*, const int*, const int*, long, int, int,
                       int, int, int, float, long, float*, int, bool,
                       const int*, int, hipStream_t);
void launch_rope_paged_attn(bf16*, const bf16*, const bf16*, const bf16*,
                            const long*, const float*, const long*, bf16*,
                            bf16*, const int*, const int*, long, int, int,
                            int, float, long, long, long, float*, int, bool,
                            hipStream_t);
void launch_attn_prefill_mfma(bf16*, const bf16*, const bf16*,
                              const bf16*, const int*, int, long, int, int,
                              int, float, long, long, long, hipStream_t);
void launch_attn_prefill_paged(bf16*, const bf16*, const bf16*, const bf16*,
                               const int*, const int*, const int*, int, long,
                               int, int, int, int, float, long, bool,
                               hipStream_t);
void launch_experts_few(bool, bf16*, int*, const bf16*, const bf16*, const int*,
                        int, int, int, int, int, hipStream_t);
template <typename T>
void launch_gelu_mul(T*, const T*, long, int, hipStream_t);
template <typename T>
void launch_embed_dyt(T*, float*, const T*, const long*, const float*,
                      const float*, const float*, long, int, long,
                      hipStream_t);
template <typename T>
void launch_add_dyt(T*, float*, const T*, const float*, const float*,
                    const float*, const float*, const float*, const float*,
                    long, int, hipStream_t);
template <typename T>
void launch_rope_pairs_append(T*, const T*, const T*, const long*,
                              const double*, const long*, T*, T*, long, int,
                              int, int, int, int, int, int, long, long, long,
                              hipStream_t);
template <typename T>
void launch_window_attn_general(T*, const T*, const T*, const T*, const int*,
                                const long*, const int*, const float*, long,
                                int, int, int, int, int, int, float, float,
                                float, long, hipStream_t);
void launch_window_attn_prefill(bf16*, const bf16*, const bf16*, const bf16*,
                                const int*, const long*, const int*,
                                const int*, const float*, int, int, int, int,
                                int, int, int, float, float, float, long,
                                hipStream_t);
void launch_window_attn_decode(bf16*, const bf16*, const bf16*, const bf16*,
                               const int*, const long*, const float*, float*,
                               long, int, int, int, int, int, int, float,
                               float, float, long, int, hipStream_t);
bool recurrent_chunk_fits(int, int, int);
void launch_gla_chunk_gates(float*, const bf16*, const bf16*, const float*,
                            const int*, const int*, int, int, int, float,
                            long, hipStream_t);
void launch_mlstm_chunk_gates(float*, float*, const float*, const float*,
                              const float*, const int*, const int*, int, int,
                              float, hipStream_t);
void launch_recurrent_chunk(Kind, bf16*, float*, float*, float*, float*,
                            float*, float*, float*, const bf16*, const bf16*, const bf16*,
                            const bf16*, const float*, const float*,
                            const float*, const int*, const long*,
                            const int*, const int*, const int*, int, int,
                            int, int, int, long, float, float, hipStream_t);
template <typename T>
void launch_gla_decay(float*, const T*, const T*, const float*, long, int,
                      int, float, long, hipStream_t);
void launch_mlstm_gates(float*, const float*, const float*, const float*,
                        long, int, float, hipStream_t);
template <typename T>
void launch_recurrent_scan(Kind, float*, float*, float*, float*, float*,
                           const T*, const T*, const T*, const float*, const int*,
                           const long*, const int*, int, int, int, int, long,
                           float, hipStream_t);
template <typename T>
void launch_recurrent_out(T*, const float*, const T*, const float*, bool,
                          long, int, int, long, float, hipStream_t);
template <typename T>
void launch_recurrent_step(Kind, T*, float*, float*, float*, float*,
                           const T*, const T*,
                           const T*, const T*, const T*, const T*,
                           const float*, const float*, const float*,
                           const float*, const long*, const int*, long, int,
                           int, int, int, long, float, float, float,
                           hipStream_t);
void launch_decode_inputs(const long*, const int*, long*, long*, long*, int*,
                          int*, int*, int, int, int, int, int, hipStream_t);
bool gemm_rows_fits(long, long);
void launch_gemm_split(bf16*, float*, const void*, const void*, const float*,
                       const float*, int, int, int, long, long, int, int, int,
                       bool, hipStream_t);
void launch_gemm_wide(bf16*, float*, const bf16*, const bf16*, int, int, int,
                      long, long, int, int, int, bool, hipStream_t);
void launch_gemm_rows(bf16*, const bf16*, const bf16*, const float*,
                      const float*, int, int, int, long, long, long,
                      hipStream_t);
void launch_silu_mul(bf16*, const bf16*, long, int, hipStream_t);
void launch_quant_fp8(unsigned char*, float*, const bf16*, long, int, long,
                      hipStream_t);
void launch_fused_add_rmsnorm_fp8(unsigned char*, float*, const bf16*,
                                  bf16*, const bf16*, float, long, int,
                                  hipStream_t);
void launch_parts_add_rmsnorm_fp8(unsigned char*, float*, const float*, int,
                                  bf16*, const bf16*, float, long, int,
                                  hipStream_t);
void launch_silu_mul_fp8(unsigned char*, float*, const bf16*, long, int,
                         hipStream_t);
void launch_moe_gemm(bf16*, float*, const bf16*, const bf16*, const int*,
                     const int*, int, int, int, int, int, hipStream_t);
template <typename T>
void launch_greedy_sample(long*, const T*, long, int, hipStream_t);
template <typename T>
void launch_sample(long*, const T*, const float*, const float*, const int*,
                   const float*, void*, long, int, hipStream_t);
long sample_workspace(long rows, int vocab);

namespace {

bf16* bf(torch::Tensor& t) { return reinterpret_cast<bf16*>(t.data_ptr()); }
const bf16* cbf(const torch::Tensor& t) {
  return reinterpret_cast<const bf16*>(t.data_ptr());
}

void rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
             double eps) {
  check(out, torch::kBFloat16, "out");
  check(x, torch::kBFloat16, "x");
  check(w, torch::kBFloat16, "w");
  const int hidden = (int)x.size(-1);
  TORCH_CHECK(hidden % 8 == 0 && hidden <= 16384, "hidden size");
  launch_rmsnorm(bf(out), cbf(x), cbf(w), (float)eps, x.numel() / hidden,
                 hidden, stream());
}

// x <- rmsnorm(residual + the sum of parts [splits, rows, hidden]) * w, and
// residual that sum, the parts' rounded first
void parts_add_rmsnorm(torch::Tensor x, torch::Tensor parts,
                       torch::Tensor residual, torch::Tensor w, double eps) {
  check(x, torch::kBFloat16, "x");
  check(parts, torch::kFloat, "parts");
  check(residual, torch::kBFloat16, "residual");
  check(w, torch::kBFloat16, "w");
  TORCH_CHECK(parts.dim() == 3 && parts.size(0) >= 2 && parts.size(0) <= 8,
              "parts_add_rmsnorm: 2 to 8 parts");
  const long rows = parts.size(1);
  const int hidden = (int)parts.size(2);
  TORCH_CHECK(hidden % 8 == 0 && hidden <= 8192 && w.numel() == hidden &&
                  x.numel() == rows * hidden && residual.numel() == x.numel(),
              "parts_add_rmsnorm: shape");
  if (rows == 0) return;
  launch_parts_add_rmsnorm(bf(x), parts.data_ptr<float>(), (int)parts.size(0),
                           bf(residual), cbf(w), (float)eps, rows, hidden,
                           stream());
}

// x <- rmsnorm(residual + y) * w and residual that sum, y the weighted sum of a
// row's choices, rows of `data`: place [rows, n], weight [rows, n]
void choices_add_rmsnorm(torch::Tensor x, torch::Tensor data,
                         torch::Tensor place, torch::Tensor weight,
                         torch::Tensor residual, torch::Tensor w, double eps) {
  check(x, torch::kBFloat16, "x");
  check(data, torch::kBFloat16, "data");
  check(place, torch::kInt32, "place");
  check(weight, torch::kFloat, "weight");
  check(residual, torch::kBFloat16, "residual");
  check(w, torch::kBFloat16, "w");
  TORCH_CHECK(data.dim() == 2 && place.dim() == 2 && place.size(1) >= 1 &&
                  weight.sizes() == place.sizes(),
              "choices_add_rmsnorm: shape");
  const long rows = place.size(0);
  const int hidden = (int)data.size(1);
  TORCH_CHECK(hidden % 8 == 0 && hidden <= 8192 && w.numel() == hidden &&
                  x.numel() == rows * hidden &&
                  residual.numel() == x.numel(),
              "choices_add_rmsnorm: shape");
  if (rows == 0) return;
  launch_choices_add_rmsnorm(bf(x), cbf(data), place.data_ptr<int>(),
                             weight.data_ptr<float>(), (int)place.size(1),
                             bf(residual), cbf(w), (float)eps, rows, hidden,
                             stream());
}

void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual,
                       torch::Tensor w, double eps) {
  check(x, torch::kBFloat16, "x");
  check(residual, torch::kBFloat16, "residual");
  const int hidden = (int)x.size(-1);
  TORCH_CHECK(hidden % 8 == 0 && hidden <= 16384, "hidden size");
  launch_fused_add_rmsnorm(bf(x), bf(residual), cbf(w), (float)eps,
                           x.numel() / hidden, hidden, stream());
}

// Products of P choices with their experts' weights w [E, 2N (up) or N, K]:
// out [P, N], x [P / div, K] (up) or [P, K], ids [P] int32; place [P] int32
// becomes p, or -1 where ids names no expert, whose row of out is left as it is
void experts_few(bool up, torch::Tensor out,
                 c10::optional<torch::Tensor> place, torch::Tensor x,
                 torch::Tensor w, torch::Tensor ids, long div) {
  check(out, torch::kBFloat16, "out");
  check(x, torch::kBFloat16, "x");
  check(w, torch::kBFloat16, "w");
  check(ids, torch::kInt32, "ids");
  TORCH_CHECK(out.dim() == 2 && x.dim() == 2 && w.dim() == 3 && div >= 1,
              "experts_few: shape");
  const long P = ids.numel(), N = out.size(1), K = x.size(1);
  TORCH_CHECK(P >= 1 && P <= 384 && out.size(0) == P &&
                  x.size(0) * (up ? div : 1) == P && w.size(2) == K &&
                  w.size(1) == (up ? 2 * N : N) && w.size(0) >= 1 &&
                  w.size(0) <= 64 && N % 128 == 0 && K % 128 == 0,
              "experts_few: shape");
  if (place.has_value()) {
    check(*place, torch::kInt32, "place");
    TORCH_CHECK(place->numel() == P, "experts_few: place");
  }
  launch_experts_few(up, bf(out),
                     place.has_value() ? place->data_ptr<int>() : nullptr,
                     cbf(x), cbf(w), ids.data_ptr<int>(), (int)P,
                     (int)w.size(0), (int)N, (int)K, (int)div, stream());
}

// q/k/v may be strided views into one fused qkv buffer: require only the
// head dim contiguous (stride(2)==1) and head stride == D.
void check_qkv_view(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == torch::kBFloat16, name, " must be bf16");
  TORCH_CHECK(t.dim() == 3 && t.stride(2) == 1 &&
                  t.stride(1) == t.size(2),
              name, " must be [T, H, D] with contiguous heads");
}

void rope_kv_append(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                    torch::Tensor positions, torch::Tensor cos_sin,
                    torch::Tensor slot_mapping, torch::Tensor k_cache,
                    torch::Tensor v_cache) {
  check_qkv_view(q, "q");
  check_qkv_view(k, "k");
  check_qkv_view(v, "v");
  check(cos_sin, torch::kFloat32, "cos_sin");
  check(positions, torch::kInt64, "positions");
  check(slot_mapping, torch::kInt64, "slot_mapping");
  const long T = q.size(0);
  const int H = (int)q.size(1), KV = (int)k.size(1), D = (int)q.size(2);
  const int BS = (int)k_cache.size(2);
  const bool kv_fp8 =
      k_cache.scalar_type() == torch::kFloat8_e4m3fn;
  launch_rope_kv_append(bf(q), bf(k), cbf(v),
                        positions.data_ptr<long>(),
                        cos_sin.data_ptr<float>(),
                        slot_mapping.data_ptr<long>(), bf(k_cache),
                        bf(v_cache), T, H, KV, D, BS, q.stride(0),
                        k.stride(0), v.stride(0), kv_fp8, stream());
}

void paged_attn(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                torch::Tensor v_cache, torch::Tensor block_tables,
                torch::Tensor ctx_lens,
                c10::optional<torch::Tensor> row_seq, double scale,
                c10::optional<torch::Tensor> split_ws, long split) {
  check(out, torch::kBFloat16, "out");
  check_qkv_view(q, "q");
  check(block_tables, torch::kInt32, "block_tables");
  check(ctx_lens, torch::kInt32, "ctx_lens");
  const long R = q.size(0);
  const int H = (int)q.size(1), D = (int)q.size(2);
  const int KV = (int)k_cache.size(1), BS = (int)k_cache.size(2);
  TORCH_CHECK(H % KV == 0, "GQA group");
  const int* rs = nullptr;
  if (row_seq.has_value()) {
    check(*row_seq, torch::kInt32, "row_seq");
    rs = row_seq->data_ptr<int>();
  }
  float* ws = nullptr;
  if (split > 1) {
    TORCH_CHECK(split_ws.has_value(), "split>1 needs a workspace");
    check(*split_ws, torch::kFloat, "split_ws");
    TORCH_CHECK(split_ws->numel() >= R * KV * split * (H / KV) * (D + 2),
                "split_ws too small");
    ws = split_ws->data_ptr<float>();
  }
  const bool kv_fp8 =
      k_cache.scalar_type() == torch::kFloat8_e4m3fn;
  TORCH_CHECK(v_cache.scalar_type() == k_cache.scalar_type(),
              "k/v cache dtype mismatch");
  launch_paged_attn(bf(out), cbf(q), cbf(k_cache), cbf(v_cache),
                    block_tables.data_ptr<int>(), ctx_lens.data_ptr<int>(),
                    rs, R, KV, H / KV, D, (int)block_tables.size(1), BS,
                    (float)scale, q.stride(0), ws, (int)split, kv_fp8,
                    nullptr, 0, stream());
}

// rope_kv_append and paged_attn in one launch; q and k stay as they are
void rope_paged_attn(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                     torch::Tensor v, torch::Tensor positions,
                     torch::Tensor cos_sin, torch::Tensor slot_mapping,
                     torch::Tensor k_cache, torch::Tensor v_cache,
                     torch::Tensor block_tables, torch::Tensor ctx_lens,
                     double scale, c10::optional<torch::Tensor> split_ws,
                     long split) {
  check(out, torch::kBFloat16, "out");
  for (const auto& t : {q, k, v}) {
    check_qkv_view(t, "q, k, v");
    TORCH_CHECK(t.stride(0) % 8 == 0 &&
                    reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
                "rope_paged_attn: rows of q, k, v must be 16-byte aligned");
  }
  check(cos_sin, torch::kFloat32, "cos_sin");
  check(positions, torch::kInt64, "positions");
  check(slot_mapping, torch::kInt64, "slot_mapping");
  check(block_tables, torch::kInt32, "block_tables");
  check(ctx_lens, torch::kInt32, "ctx_lens");
  const long R = q.size(0);
  const int H = (int)q.size(1), KV = (int)k.size(1);
  TORCH_CHECK(KV > 0 && H % KV == 0, "GQA group");
  const int group = H / KV;
  TORCH_CHECK(group <= 4 || group == 8, "rope_paged_attn: group");
  for (const auto& t : {k_cache, v_cache})
    TORCH_CHECK(t.is_cuda() && t.is_contiguous() && t.dim() == 4 &&
                    t.size(1) == KV && t.size(2) == 16 && t.size(3) == 128 &&
                    t.scalar_type() == k_cache.scalar_type(),
                "rope_paged_attn: k/v cache");
  const bool kv_fp8 = k_cache.scalar_type() == torch::kFloat8_e4m3fn;
  TORCH_CHECK(kv_fp8 || k_cache.scalar_type() == torch::kBFloat16,
              "rope_paged_attn: k/v cache dtype");
  TORCH_CHECK(q.size(2) == 128 && k.size(2) == 128 && v.size(2) == 128 &&
                  k.size(0) == R && v.size(0) == R && v.size(1) == KV &&
                  out.numel() == q.numel() && cos_sin.size(-1) == 128,
              "rope_paged_attn: shape");
  TORCH_CHECK(positions.numel() >= R && slot_mapping.numel() >= R &&
                  ctx_lens.numel() >= R && block_tables.dim() == 2 &&
                  block_tables.size(0) >= R, "rope_paged_attn: rows");
  TORCH_CHECK(split >= 1 && split <= 64, "rope_paged_attn: 1 to 64 parts");
  float* ws = nullptr;
  if (split > 1) {
    TORCH_CHECK(split_ws.has_value(), "split>1 needs a workspace");
    check(*split_ws, torch::kFloat, "split_ws");
    TORCH_CHECK(split_ws->numel() >= R * split * H * 130,
                "split_ws too small");
    ws = split_ws->data_ptr<float>();
  }
  launch_rope_paged_attn(
      bf(out), cbf(q), cbf(k), cbf(v), positions.data_ptr<long>(),
      cos_sin.data_ptr<float>(), slot_mapping.data_ptr<long>(), bf(k_cache),
      bf(v_cache), block_tables.data_ptr<int>(), ctx_lens.data_ptr<int>(), R,
      KV, group, (int)block_tables.size(1), (float)scale, q.stride(0),
      k.stride(0), v.stride(0), ws, (int)split, kv_fp8, stream());
}

void attn_prefill_mfma(torch::Tensor out, torch::Tensor q, torch::Tensor k,
                       torch::Tensor v, torch::Tensor seq_start,
                       long /*max_seqlen*/, double scale) {
  check(out, torch::kBFloat16, "out");
  check_qkv_view(q, "q");
  check_qkv_view(k, "k");
  check_qkv_view(v, "v");
  check(seq_start, torch::kInt32, "seq_start");
  TORCH_CHECK(seq_start.numel() >= 1, "seq_start");
  const int H = (int)q.size(1), D = (int)q.size(2);
  const int KV = (int)k.size(1);
  TORCH_CHECK(KV > 0 && H % KV == 0, "GQA group");
  // keys and values are read 16 bytes at a time straight into LDS, the rows of a
  // tile by 32 bits of offset
  auto aligned = [](const torch::Tensor& t) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 &&
                   t.stride(0) % 8 == 0 && t.stride(0) < (1l << 25)
               ? t : t.clone(at::MemoryFormat::Contiguous);
  };
  k = aligned(k);
  v = aligned(v);
  launch_attn_prefill_mfma(
      bf(out), cbf(q), cbf(k), cbf(v), seq_start.data_ptr<int>(),
      (int)seq_start.numel() - 1, q.size(0), H, KV, D, (float)scale,
      q.stride(0), k.stride(0), v.stride(0), stream());
}

// Attention of portions over the pages, head_dim 128: on the matrix cores from
// min_rows rows on; with `short_too` the rows of shorter ones one by one.
void attn_portions(torch::Tensor out, torch::Tensor q, torch::Tensor k_cache,
                   torch::Tensor v_cache, torch::Tensor block_tables,
                   torch::Tensor ctx_lens, torch::Tensor row_seq,
                   torch::Tensor seq_start, long min_rows, bool short_too,
                   double scale) {
  check(out, torch::kBFloat16, "out");
  check_qkv_view(q, "q");
  check(block_tables, torch::kInt32, "block_tables");
  check(ctx_lens, torch::kInt32, "ctx_lens");
  check(row_seq, torch::kInt32, "row_seq");
  check(seq_start, torch::kInt32, "seq_start");
  const long T = q.size(0), seqs = seq_start.numel() - 1;
  const int H = (int)q.size(1), KV = (int)k_cache.size(1);
  const int max_blocks = (int)block_tables.size(1);
  TORCH_CHECK(KV > 0 && H % KV == 0, "GQA group");
  TORCH_CHECK(q.size(2) == 128 && k_cache.size(3) == 128 &&
                  k_cache.size(2) == 16, "attn_portions: shape");
  TORCH_CHECK(v_cache.scalar_type() == k_cache.scalar_type() &&
                  k_cache.is_contiguous() && v_cache.is_contiguous(),
              "k/v cache");
  TORCH_CHECK(ctx_lens.numel() >= T && row_seq.numel() >= T &&
                  block_tables.size(0) >= seqs, "attn_portions: rows");
  const bool fp8 = k_cache.scalar_type() == torch::kFloat8_e4m3fn;
  if (short_too)
    launch_paged_attn(bf(out), cbf(q), cbf(k_cache), cbf(v_cache),
                      block_tables.data_ptr<int>(), ctx_lens.data_ptr<int>(),
                      row_seq.data_ptr<int>(), T, KV, H / KV, 128, max_blocks,
                      16, (float)scale, q.stride(0), nullptr, 1, fp8,
                      seq_start.data_ptr<int>(), (int)min_rows - 1, stream());
  launch_attn_prefill_paged(
      bf(out), cbf(q), cbf(k_cache), cbf(v_cache),
      block_tables.data_ptr<int>(), ctx_lens.data_ptr<int>(),
      seq_start.data_ptr<int>(), (int)seqs, T, H, KV, max_blocks,
      (int)min_rows, (float)scale, q.stride(0), fp8, stream());
}

// stage: long [5 * cap], then int [B, staged] page ids
void decode_inputs(torch::Tensor stage, long B, long cap, long staged,
                   torch::Tensor ids, torch::Tensor positions,
                   torch::Tensor slots, torch::Tensor lens,
                   c10::optional<torch::Tensor> state, torch::Tensor tables) {
  check(stage, torch::kLong, "stage");
  for (const auto& t : {ids, positions, slots}) check(t, torch::kLong, "ids");
  check(lens, torch::kInt32, "lens");
  check(tables, torch::kInt32, "tables");
  if (state.has_value()) check(*state, torch::kInt32, "state");
  const long bucket = ids.numel();
  TORCH_CHECK(tables.dim() == 2 && tables.size(0) == bucket &&
                  positions.numel() == bucket && slots.numel() == bucket &&
                  lens.numel() == bucket &&
                  (!state.has_value() || state->numel() == bucket),
              "decode_inputs: rows");
  TORCH_CHECK(B >= 0 && B <= bucket && B <= cap && staged >= 0 &&
                  staged <= tables.size(1) &&
                  stage.numel() * 8 >= cap * 40 + B * staged * 4,
              "decode_inputs: sizes");
  long* s = stage.data_ptr<long>();
  launch_decode_inputs(s, reinterpret_cast<int*>(s + 5 * cap),
                       ids.data_ptr<long>(), positions.data_ptr<long>(),
                       slots.data_ptr<long>(), lens.data_ptr<int>(),
                       state.has_value() ? state->data_ptr<int>() : nullptr,
                       tables.data_ptr<int>(), (int)B, (int)bucket, (int)cap,
                       (int)staged, (int)tables.size(1), stream());
}

// out = x w^T; with scales of the rows x and w are e4m3
void gemm_rows(torch::Tensor out, torch::Tensor x, torch::Tensor w,
               c10::optional<torch::Tensor> x_scale,
               c10::optional<torch::Tensor> w_scale) {
  const bool fp8 = x_scale.has_value();
  const auto kind = fp8 ? torch::kFloat8_e4m3fn : torch::kBFloat16;
  for (const auto& t : {out, x, w})
    TORCH_CHECK(t.is_cuda() && t.dim() == 2 && t.stride(1) == 1,
                "gemm_rows: matrices");
  TORCH_CHECK(out.scalar_type() == torch::kBFloat16 &&
                  x.scalar_type() == kind && w.scalar_type() == kind &&
                  w_scale.has_value() == fp8, "gemm_rows: matrices");
  const long M = x.size(0), N = w.size(0), per = fp8 ? 2 : 1;
  const long K = x.size(1) / per;            // units of 2 bytes
  TORCH_CHECK(w.size(1) == x.size(1) && x.size(1) % per == 0 &&
                  out.size(0) == M && out.size(1) == N, "gemm_rows: shape");
  auto aligned = [](const torch::Tensor& t, long n) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % (2 * n) == 0 &&
           t.stride(0) * t.element_size() % (2 * n) == 0;
  };
  if (fp8) {
    check(*x_scale, torch::kFloat, "x_scale");
    check(*w_scale, torch::kFloat, "w_scale");
    TORCH_CHECK(x_scale->numel() == M && w_scale->numel() == N &&
                    reinterpret_cast<uintptr_t>(w_scale->data_ptr()) % 16 == 0,
                "gemm_rows: scales");
  }
  TORCH_CHECK(gemm_rows_fits(M, K) && N % 4 == 0 && K % 8 == 0 &&
                  N < (1l << 31) && aligned(x, 8) && aligned(w, 8) &&
                  aligned(out, 4), "gemm_rows: sizes");
  if (N == 0) return;
  launch_gemm_rows(bf(out), cbf(x), cbf(w),
                   fp8 ? x_scale->data_ptr<float>() : nullptr,
                   fp8 ? w_scale->data_ptr<float>() : nullptr, (int)M, (int)N,
                   (int)K, x.stride(0) / per, w.stride(0) / per, out.stride(0),
                   stream());
}

// out = x w^T, K in `splits` parts that a second kernel adds up; without out
// the parts, [splits, M, N] floats, are the result.  With scales of the rows x
// and w are e4m3.  gated: out = silu(gate) * up of the halves of w.
void gemm_split(c10::optional<torch::Tensor> out, torch::Tensor x,
                torch::Tensor w, c10::optional<torch::Tensor> part, long bm,
                long bn, long splits, c10::optional<torch::Tensor> x_scale,
                c10::optional<torch::Tensor> w_scale, bool gated) {
  const bool fp8 = x_scale.has_value();
  const auto kind = fp8 ? torch::kFloat8_e4m3fn : torch::kBFloat16;
  for (const auto& t : {x, w})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == kind && t.dim() == 2 &&
                    t.stride(1) == 1, "gemm_split: matrices");
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K && (out.has_value() || splits > 1) &&
                  w_scale.has_value() == fp8, "gemm_split: shape");
  if (fp8) {
    check(*x_scale, torch::kFloat, "x_scale");
    check(*w_scale, torch::kFloat, "w_scale");
    TORCH_CHECK(x_scale->numel() == M && w_scale->numel() == N &&
                    reinterpret_cast<uintptr_t>(w_scale->data_ptr()) % 16 == 0,
                "gemm_split: scales");
  }
  if (out.has_value())
    TORCH_CHECK(out->is_cuda() && out->scalar_type() == torch::kBFloat16 &&
                    out->dim() == 2 && out->size(0) == M &&
                    out->size(1) == (gated ? N / 2 : N) &&
                    out->is_contiguous() &&
                    reinterpret_cast<uintptr_t>(out->data_ptr()) % 8 == 0,
                "gemm_split: out");
  const long unit = fp8 ? 16 : 8, chunk = fp8 ? 256 : 128;
  // 16 bytes at a time, the rows of a tile by 32 bits of offset
  auto fits = [&](const torch::Tensor& t, long rows) {
    const long reach = (std::min(t.size(0), rows) - 1) * t.stride(0) + K;
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 &&
           t.stride(0) % unit == 0 && reach < 0xfffffff0l / (fp8 ? 1 : 2);
  };
  TORCH_CHECK(N % 4 == 0 && K % chunk == 0 && K >= chunk && M < (1l << 20) &&
                  K < (1l << 24) && N < (1l << 24) && fits(x, bm) &&
                  fits(w, bn), "gemm_split: sizes");
  TORCH_CHECK(fp8 ? bm == 64 && (bn == 32 || bn == 64 || bn == 128)
                  : ((bm == 64 || bm == 128) && (bn == 64 || bn == 128)) ||
                        (bm == 256 && bn == 128), "gemm_split: tile");
  if (gated)      // 32 bits of offset reach the up rows
    TORCH_CHECK(!fp8 && splits == 1 && N % 8 == 0 &&
                    (N / 2 + 128) * w.stride(0) < (1l << 31),
                "gemm_split: gated");
  TORCH_CHECK(splits >= 1 && splits <= 8 && splits <= K / chunk,
              "gemm_split: 1 to 8 parts");
  float* ws = nullptr;
  if (splits > 1) {
    TORCH_CHECK(part.has_value(), "gemm_split: parts need a workspace");
    check(*part, torch::kFloat, "part");
    TORCH_CHECK(part->numel() >= splits * M * N, "gemm_split: workspace");
    ws = part->data_ptr<float>();
  }
  if (M == 0 || N == 0) return;
  launch_gemm_split(out.has_value() ? bf(*out) : nullptr, ws, x.data_ptr(),
                    w.data_ptr(), fp8 ? x_scale->data_ptr<float>() : nullptr,
                    fp8 ? w_scale->data_ptr<float>() : nullptr, (int)M, (int)N,
                    (int)K, x.stride(0), w.stride(0), (int)bm, (int)bn,
                    (int)splits, gated, stream());
}

// products of many rows in tiles of 32 * high by bn: out, or the parts
void gemm_wide(c10::optional<torch::Tensor> out, torch::Tensor x,
               torch::Tensor w, c10::optional<torch::Tensor> part, long high,
               long bn, long splits, bool gated) {
  for (const auto& t : {x, w})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16 &&
                    t.dim() == 2 && t.stride(1) == 1, "gemm_wide: matrices");
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  const long outs = gated ? N / 2 : N;
  TORCH_CHECK(w.size(1) == K && out.has_value() != (splits > 1) &&
                  !(gated && splits > 1), "gemm_wide: shape");
  if (out.has_value())
    TORCH_CHECK(out->is_cuda() && out->scalar_type() == torch::kBFloat16 &&
                    out->dim() == 2 && out->size(0) == M &&
                    out->size(1) == outs && out->is_contiguous() &&
                    reinterpret_cast<uintptr_t>(out->data_ptr()) % 16 == 0,
                "gemm_wide: out");
  TORCH_CHECK(high >= 4 && high <= 8 && (bn == 128 || bn == 256) &&
                  splits >= 1 && splits <= 8 && K >= 64 * splits &&
                  K % 64 == 0 && N % (gated ? 16 : 8) == 0,
              "gemm_wide: sizes");
  // 16 bytes at a time, the rows of a tile by 32 bits of offset
  auto fits = [&](const torch::Tensor& t, long rows) {
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 &&
           t.stride(0) % 8 == 0 && t.stride(0) >= 0 &&
           (rows - 1) * t.stride(0) + K < 0x7ffffff8l;
  };
  const long tiles = (M / (32 * high) + 1) * (outs / 64 + 1) * splits;
  TORCH_CHECK(fits(x, std::min(M, 32 * high)) &&
                  fits(w, gated ? std::min(N, outs + 128) : std::min(N, bn)) &&
                  tiles < (1l << 30), "gemm_wide: offsets");
  float* ws = nullptr;
  if (splits > 1) {
    TORCH_CHECK(part.has_value(), "gemm_wide: parts need a workspace");
    check(*part, torch::kFloat, "part");
    TORCH_CHECK(part->numel() >= splits * M * N, "gemm_wide: workspace");
    ws = part->data_ptr<float>();
  }
  if (M == 0 || N == 0) return;
  launch_gemm_wide(out.has_value() ? bf(*out) : nullptr, ws, cbf(x), cbf(w),
                   (int)M, (int)N, (int)K, x.stride(0), w.stride(0), (int)high,
                   (int)bn, (int)splits, gated, stream());
}

void silu_mul(torch::Tensor out, torch::Tensor x) {
  check(out, torch::kBFloat16, "out");
  check(x, torch::kBFloat16, "x");
  const int inter = (int)out.size(-1);
  TORCH_CHECK(x.size(-1) == 2 * inter && inter % 8 == 0, "shape");
  launch_silu_mul(bf(out), cbf(x), out.numel() / inter, inter, stream());
}

// ---- bf16 | float kernels ------------------------------------------------

void check_dyt(const torch::Tensor& w, const torch::Tensor& b,
               const torch::Tensor& a, long width) {
  check_param(w, width, "norm weight");
  check_param(b, width, "norm bias");
  check_param(a, 1, "norm alpha");
}

void gelu_mul(torch::Tensor out, torch::Tensor x) {
  check(out, x.scalar_type(), "out");
  check(x, x.scalar_type(), "x");
  const long inter = out.size(-1);
  TORCH_CHECK(x.size(-1) == 2 * inter &&
              x.numel() == 2 * out.numel(), "gelu_mul: shape");
  by_dtype(x, [&](auto tag) {
    using T = ELEM(tag);
    launch_gelu_mul<T>(ptr<T>(out), ptr<T>(x), out.numel() / inter,
                       (int)inter, stream());
  });
}

void embed_dyt(torch::Tensor out, torch::Tensor residual,
               torch::Tensor table, torch::Tensor ids, torch::Tensor w,
               torch::Tensor b, torch::Tensor a) {
  const long rows = ids.numel(), width = table.size(1);
  check(table, table.scalar_type(), "table");
  check(out, table.scalar_type(), "out");
  check(residual, torch::kFloat32, "residual");
  check(ids, torch::kInt64, "ids");
  check_dyt(w, b, a, width);
  TORCH_CHECK(out.numel() == rows * width &&
              residual.numel() == rows * width, "embed_dyt: shape");
  by_dtype(table, [&](auto tag) {
    using T = ELEM(tag);
    launch_embed_dyt<T>(ptr<T>(out), ptr<float>(residual), ptr<T>(table),
                        ids.data_ptr<long>(), ptr<float>(w), ptr<float>(b),
                        ptr<float>(a), rows, (int)width, table.size(0),
                        stream());
  });
}

void add_dyt(c10::optional<torch::Tensor> out, torch::Tensor residual,
             torch::Tensor h, torch::Tensor w1, torch::Tensor b1,
             torch::Tensor a1, torch::Tensor w2, torch::Tensor b2,
             torch::Tensor a2) {
  const long width = h.size(-1), rows = h.numel() / width;
  check(h, h.scalar_type(), "h");
  check(residual, torch::kFloat32, "residual");
  check_dyt(w1, b1, a1, width);
  check_dyt(w2, b2, a2, width);
  TORCH_CHECK(residual.numel() == h.numel(), "add_dyt: shape");
  if (out.has_value()) {
    check(*out, h.scalar_type(), "out");
    TORCH_CHECK(out->numel() == h.numel(), "add_dyt: shape");
  }
  by_dtype(h, [&](auto tag) {
    using T = ELEM(tag);
    launch_add_dyt<T>(out.has_value() ? ptr<T>(*out) : nullptr,
                      ptr<float>(residual), ptr<T>(h), ptr<float>(w1),
                      ptr<float>(b1), ptr<float>(a1), ptr<float>(w2),
                      ptr<float>(b2), ptr<float>(a2), rows, (int)width,
                      stream());
  });
}

// shapes of the transposed-V paged cache; returns {G, MD, E, BS}
std::array<int, 4> check_window_cache(const torch::Tensor& k_cache,
                                      const torch::Tensor& v_cache,
                                      torch::ScalarType dt) {
  check(k_cache, dt, "k_cache");
  check(v_cache, dt, "v_cache");
  TORCH_CHECK(k_cache.dim() == 4 && v_cache.dim() == 4 &&
                  k_cache.size(0) == v_cache.size(0) &&
                  k_cache.size(1) == v_cache.size(1) &&
                  k_cache.size(2) == v_cache.size(3),
              "window cache: k [NB, G, BS, 2D], v [NB, G, E, BS]");
  return {(int)k_cache.size(1), (int)k_cache.size(3),
          (int)v_cache.size(2), (int)k_cache.size(2)};
}

void rope_pairs_append(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                       torch::Tensor positions, torch::Tensor freqs,
                       torch::Tensor slot_mapping, torch::Tensor k_cache,
                       torch::Tensor v_cache, long head_dim) {
  const auto dt = q.scalar_type();
  const auto [G, MD, E, BS] = check_window_cache(k_cache, v_cache, dt);
  const long rows = q.size(0), D = head_dim;
  TORCH_CHECK(q.dim() == 2 && q.size(1) % D == 0 && MD % D == 0,
              "rope_pairs_append: head_dim");
  check_rows(q, dt, rows, q.size(1), q.stride(0), "q");
  check_rows(k, dt, rows, (long)G * MD, k.stride(0), "k");
  check_rows(v, dt, rows, (long)G * E, v.stride(0), "v");
  check(positions, torch::kInt64, "positions");
  check(slot_mapping, torch::kInt64, "slot_mapping");
  check(freqs, torch::kFloat64, "freqs");
  TORCH_CHECK(positions.numel() == rows && slot_mapping.numel() == rows,
              "rope_pairs_append: rows");
  TORCH_CHECK(2 * freqs.numel() <= D && D <= 4096,
              "rope_pairs_append: rotary dimensions");
  by_dtype(q, [&](auto tag) {
    using T = ELEM(tag);
    launch_rope_pairs_append<T>(
        ptr<T>(q), ptr<T>(k), ptr<T>(v), positions.data_ptr<long>(),
        ptr<double>(freqs), slot_mapping.data_ptr<long>(), ptr<T>(k_cache),
        ptr<T>(v_cache), rows, (int)(q.size(1) / D), G * MD / (int)D, (int)D,
        G, E, 2 * (int)freqs.numel(), BS, q.stride(0), k.stride(0),
        v.stride(0), stream());
  });
}

void window_attn_general(torch::Tensor out, torch::Tensor q,
                         torch::Tensor k_cache, torch::Tensor v_cache,
                         torch::Tensor block_tables, torch::Tensor positions,
                         c10::optional<torch::Tensor> row_seq,
                         torch::Tensor lam, long window, double scale,
                         double diff, double eps) {
  const auto dt = q.scalar_type();
  const auto [G, MD, E, BS] = check_window_cache(k_cache, v_cache, dt);
  const long rows = q.size(0), D = MD / 2;
  TORCH_CHECK(BS == 16 && MD % 2 == 0 && E <= 1024 && D <= 4096 &&
              window >= 1, "window_attn: sizes");
  TORCH_CHECK(q.dim() == 2 && q.size(1) % MD == 0, "window_attn: q");
  const long H = q.size(1) / MD;
  TORCH_CHECK(H % G == 0, "window_attn: head groups");
  check_rows(q, dt, rows, H * MD, q.stride(0), "q");
  check(out, dt, "out");
  TORCH_CHECK(out.numel() == rows * H * E, "window_attn: out");
  check(block_tables, torch::kInt32, "block_tables");
  check(positions, torch::kInt64, "positions");
  TORCH_CHECK(positions.numel() == rows, "window_attn: rows");
  check_param(lam, 4 * D, "lam");
  const int* rs = nullptr;
  if (row_seq.has_value()) {
    check(*row_seq, torch::kInt32, "row_seq");
    TORCH_CHECK(row_seq->numel() == rows, "window_attn: row_seq");
    rs = row_seq->data_ptr<int>();
  } else {
    TORCH_CHECK(block_tables.size(0) >= rows, "window_attn: block_tables");
  }
  by_dtype(q, [&](auto tag) {
    using T = ELEM(tag);
    launch_window_attn_general<T>(
        ptr<T>(out), ptr<T>(q), ptr<T>(k_cache), ptr<T>(v_cache),
        block_tables.data_ptr<int>(), positions.data_ptr<long>(), rs,
        ptr<float>(lam), rows, (int)block_tables.size(1), (int)H, G, (int)D,
        E, (int)window, (float)scale, (float)diff, (float)eps, q.stride(0),
        stream());
  });
}

// 16-byte loads of q (rows and base), sizes of the padded kernels
bool window_attn_fits(torch::Tensor q, torch::Tensor k_cache,
                      torch::Tensor v_cache) {
  const long D = k_cache.size(3) / 2, E = v_cache.size(2);
  return q.scalar_type() == torch::kBFloat16 && D % 8 == 0 && E % 8 == 0 &&
         D <= 128 && E <= 256 && k_cache.size(3) == 2 * D &&
         q.stride(0) % 8 == 0 &&
         reinterpret_cast<uintptr_t>(q.data_ptr()) % 16 == 0;
}

struct WindowDims { int H, G, D, E; };

WindowDims check_window_fast(const torch::Tensor& out, const torch::Tensor& q,
                             const torch::Tensor& k_cache,
                             const torch::Tensor& v_cache,
                             const torch::Tensor& block_tables,
                             const torch::Tensor& positions,
                             const torch::Tensor& lam, long window) {
  const auto [G, MD, E, BS] =
      check_window_cache(k_cache, v_cache, torch::kBFloat16);
  TORCH_CHECK(window_attn_fits(q, k_cache, v_cache), "window_attn: sizes");
  const long rows = q.size(0);
  TORCH_CHECK(BS == 16 && window >= 1 && q.dim() == 2 &&
                  q.size(1) % ((long)MD * G) == 0, "window_attn: q");
  const int H = (int)(q.size(1) / MD);
  check_rows(q, torch::kBFloat16, rows, (long)H * MD, q.stride(0), "q");
  check(out, torch::kBFloat16, "out");
  TORCH_CHECK(out.numel() == rows * H * E, "window_attn: out");
  check(block_tables, torch::kInt32, "block_tables");
  check(positions, torch::kInt64, "positions");
  TORCH_CHECK(positions.numel() == rows, "window_attn: rows");
  check_param(lam, 2 * MD, "lam");
  return {H, G, MD / 2, E};
}

void window_attn_prefill(torch::Tensor out, torch::Tensor q,
                         torch::Tensor k_cache, torch::Tensor v_cache,
                         torch::Tensor block_tables, torch::Tensor positions,
                         torch::Tensor seq_start, torch::Tensor tiles,
                         torch::Tensor lam, long window, double scale,
                         double diff, double eps) {
  const auto d = check_window_fast(out, q, k_cache, v_cache, block_tables,
                                   positions, lam, window);
  check_tiles(tiles, seq_start, block_tables.size(0));
  launch_window_attn_prefill(
      bf(out), cbf(q), cbf(k_cache), cbf(v_cache),
      block_tables.data_ptr<int>(), positions.data_ptr<long>(),
      seq_start.data_ptr<int>(), tiles.data_ptr<int>(), ptr<float>(lam),
      (int)tiles.size(0), (int)block_tables.size(1), d.H, d.G, d.D, d.E,
      (int)window, (float)scale, (float)diff, (float)eps, q.stride(0),
      stream());
}

void window_attn_decode(torch::Tensor out, torch::Tensor q,
                        torch::Tensor k_cache, torch::Tensor v_cache,
                        torch::Tensor block_tables, torch::Tensor positions,
                        torch::Tensor lam,
                        c10::optional<torch::Tensor> partial, long split,
                        long window, double scale, double diff, double eps) {
  const auto d = check_window_fast(out, q, k_cache, v_cache, block_tables,
                                   positions, lam, window);
  const long rows = q.size(0);
  TORCH_CHECK(block_tables.size(0) >= rows && split >= 1 && split <= 64,
              "window_attn_decode: rows, split");
  if (split > 1) {
    TORCH_CHECK(partial.has_value(), "window_attn_decode: partial");
    check_param(*partial, rows * d.H * split * 2 * (d.E + 2), "partial");
  }
  launch_window_attn_decode(
      bf(out), cbf(q), cbf(k_cache), cbf(v_cache),
      block_tables.data_ptr<int>(), positions.data_ptr<long>(),
      ptr<float>(lam), split > 1 ? ptr<float>(*partial) : nullptr, rows,
      (int)block_tables.size(1), d.H, d.G, d.D, d.E, (int)window,
      (float)scale, (float)diff, (float)eps, q.stride(0), (int)split,
      stream());
}

void gla_decay(torch::Tensor log_decay, torch::Tensor a1h, torch::Tensor a2,
               torch::Tensor a2b, double tau) {
  const auto dt = a1h.scalar_type();
  const long rows = a1h.size(0), C = a2.size(0), R = a2.size(1);
  check_rows(a1h, dt, rows, R, a1h.stride(0), "a1h");
  check(a2, dt, "a2");
  check_param(a2b, C, "a2 bias");
  check_param(log_decay, rows * C, "log_decay");
  by_dtype(a1h, [&](auto tag) {
    using T = ELEM(tag);
    launch_gla_decay<T>(ptr<float>(log_decay), ptr<T>(a1h), ptr<T>(a2),
                        ptr<float>(a2b), rows, (int)C, (int)R, (float)tau,
                        a1h.stride(0), stream());
  });
}

void mlstm_gates(torch::Tensor out, torch::Tensor raw, torch::Tensor ib,
                 torch::Tensor fb, double cap) {
  const long H = ib.numel(), rows = raw.size(0);
  check_param(raw, rows * 2 * H, "raw gates");
  check_param(out, rows * 2 * H, "gates");
  check_param(ib, H, "input gate bias");
  check_param(fb, H, "forget gate bias");
  launch_mlstm_gates(ptr<float>(out), ptr<float>(raw), ptr<float>(ib),
                     ptr<float>(fb), rows, (int)H, (float)cap, stream());
}

struct StateDims { long slots, H, D, E; };

// S [slots, H, D, E]; n [slots, H, D] and m [slots, H] come together
StateDims check_state(const torch::Tensor& S,
                      const c10::optional<torch::Tensor>& n,
                      const c10::optional<torch::Tensor>& m) {
  check(S, torch::kFloat32, "state");
  TORCH_CHECK(S.dim() == 4 && S.size(2) <= 1024 && S.size(3) <= 1024,
              "state must be [slots, H, D <= 1024, E <= 1024]");
  TORCH_CHECK(n.has_value() == m.has_value(), "state: n and m");
  if (n.has_value()) {
    check_param(*n, S.size(0) * S.size(1) * S.size(2), "state n");
    check_param(*m, S.size(0) * S.size(1), "state m");
  }
  return {S.size(0), S.size(1), S.size(2), S.size(3)};
}

void recurrent_scan(torch::Tensor o, torch::Tensor S,
                    c10::optional<torch::Tensor> n,
                    c10::optional<torch::Tensor> m,
                    c10::optional<torch::Tensor> nm_new, torch::Tensor q,
                    torch::Tensor k, torch::Tensor v, torch::Tensor gates,
                    torch::Tensor seq_start, torch::Tensor positions,
                    torch::Tensor slots, double qscale) {
  const auto dt = q.scalar_type();
  const auto d = check_state(S, n, m);
  const long rows = q.size(0), B = slots.numel(), st = q.stride(0);
  check_rows(q, dt, rows, d.H * d.D, st, "q");
  check_rows(k, dt, rows, d.H * d.D, st, "k");
  check_rows(v, dt, rows, d.H * d.E, st, "v");
  check_param(o, rows * d.H * d.E, "o");
  check_param(gates, rows * d.H * (n.has_value() ? 2 : d.D), "gates");
  check(seq_start, torch::kInt32, "seq_start");
  check(positions, torch::kInt64, "positions");
  check(slots, torch::kInt32, "slots");
  TORCH_CHECK(seq_start.numel() == B + 1 && positions.numel() == rows &&
              B <= 65535, "recurrent_scan: sequences");
  if (n.has_value()) {
    TORCH_CHECK(nm_new.has_value(), "recurrent_scan: nm_new");
    check_param(*nm_new, B * d.H * (d.D + 1), "nm_new");
  }
  by_dtype(q, [&](auto tag) {
    using T = ELEM(tag);
    launch_recurrent_scan<T>(
        n.has_value() ? MLSTM : GLA, ptr<float>(o), ptr<float>(S), opt(n),
        opt(m), opt(nm_new), ptr<T>(q),
        ptr<T>(k), ptr<T>(v), ptr<float>(gates), seq_start.data_ptr<int>(),
        positions.data_ptr<long>(), slots.data_ptr<int>(), (int)B, (int)d.H,
        (int)d.D, (int)d.E, st, (float)qscale, stream());
  });
}

void gla_chunk_gates(torch::Tensor b, torch::Tensor a1h, torch::Tensor a2,
                     torch::Tensor a2b, torch::Tensor seq_start,
                     torch::Tensor tiles, double tau) {
  const long rows = a1h.size(0), Cn = a2.size(0), R = a2.size(1);
  check_rows(a1h, torch::kBFloat16, rows, R, a1h.stride(0), "a1h");
  check(a2, torch::kBFloat16, "a2");
  check_param(a2b, Cn, "a2 bias");
  check_param(b, rows * Cn, "b");
  check_tiles(tiles, seq_start, seq_start.numel() - 1);
  launch_gla_chunk_gates(ptr<float>(b), cbf(a1h), cbf(a2), ptr<float>(a2b),
                         seq_start.data_ptr<int>(), tiles.data_ptr<int>(),
                         (int)tiles.size(0), (int)Cn, (int)R, (float)tau,
                         a1h.stride(0), stream());
}

void mlstm_chunk_gates(torch::Tensor gates, torch::Tensor info,
                       torch::Tensor raw, torch::Tensor ib, torch::Tensor fb,
                       torch::Tensor seq_start, torch::Tensor tiles,
                       double cap) {
  const long H = ib.numel(), rows = raw.size(0);
  check_param(raw, rows * 2 * H, "raw gates");
  check_param(gates, rows * 2 * H, "gates");
  check_param(ib, H, "input gate bias");
  check_param(fb, H, "forget gate bias");
  check_tiles(tiles, seq_start, seq_start.numel() - 1);
  check_param(info, tiles.size(0) * H * 2, "info");
  launch_mlstm_chunk_gates(ptr<float>(gates), ptr<float>(info),
                           ptr<float>(raw), ptr<float>(ib), ptr<float>(fb),
                           seq_start.data_ptr<int>(), tiles.data_ptr<int>(),
                           (int)tiles.size(0), (int)H, (float)cap, stream());
}

// 16-byte loads of q, k, v, g and float4 rows of the states
bool chunk_fits(torch::Tensor S, torch::Tensor q, torch::Tensor k,
                torch::Tensor v, torch::Tensor g, long rank) {
  auto aligned = [](const torch::Tensor& t) {
    return t.scalar_type() == torch::kBFloat16 && t.stride(0) % 8 == 0 &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  return aligned(q) && aligned(k) && aligned(v) && aligned(g) &&
         recurrent_chunk_fits((int)S.size(2), (int)S.size(3), (int)rank);
}

void recurrent_chunk(torch::Tensor y, torch::Tensor U,
                     c10::optional<torch::Tensor> nU,
                     c10::optional<torch::Tensor> m_in, torch::Tensor S,
                     c10::optional<torch::Tensor> n,
                     c10::optional<torch::Tensor> m, torch::Tensor q,
                     torch::Tensor k, torch::Tensor v, torch::Tensor g,
                     torch::Tensor gates, c10::optional<torch::Tensor> info,
                     torch::Tensor w, torch::Tensor seq_start,
                     torch::Tensor positions, torch::Tensor slots,
                     torch::Tensor tiles, torch::Tensor tile_start,
                     double qscale, double eps) {
  const auto d = check_state(S, n, m);
  const auto dt = torch::kBFloat16;
  const long rows = q.size(0), st = q.stride(0), B = slots.numel();
  const bool mlstm = n.has_value();
  TORCH_CHECK(chunk_fits(S, q, k, v, g, 1), "recurrent_chunk: sizes");
  check_rows(q, dt, rows, d.H * d.D, st, "q");
  check_rows(k, dt, rows, d.H * d.D, st, "k");
  check_rows(v, dt, rows, d.H * d.E, st, "v");
  check_rows(g, dt, rows, d.H * d.E, st, "g");
  check(y, dt, "y");
  TORCH_CHECK(y.numel() == rows * d.H * d.E, "recurrent_chunk: y");
  check(positions, torch::kInt64, "positions");
  check(slots, torch::kInt32, "slots");
  check(tile_start, torch::kInt32, "tile_start");
  check_tiles(tiles, seq_start, B);
  const long nt = tiles.size(0);
  TORCH_CHECK(positions.numel() == rows && tile_start.numel() == B + 1 &&
                  B <= 65535, "recurrent_chunk: sequences");
  check_param(U, nt * d.H * d.D * d.E, "U");
  check_param(gates, rows * d.H * (mlstm ? 2 : d.D), "gates");
  check_param(w, mlstm ? d.H * d.E : d.E, "norm weight");
  if (mlstm) {
    TORCH_CHECK(nU.has_value() && m_in.has_value() && info.has_value(),
                "recurrent_chunk: scratch");
    check_param(*nU, nt * d.H * d.D, "nU");
    check_param(*m_in, nt * d.H, "m_in");
    check_param(*info, nt * d.H * 2, "info");
  }
  launch_recurrent_chunk(
      mlstm ? MLSTM : GLA, bf(y), nullptr, ptr<float>(U), opt(nU),
      opt(m_in), ptr<float>(S), opt(n),
      opt(m), cbf(q), cbf(k), cbf(v), cbf(g), ptr<float>(gates), opt(info),
      ptr<float>(w), seq_start.data_ptr<int>(), positions.data_ptr<long>(),
      slots.data_ptr<int>(), tiles.data_ptr<int>(),
      tile_start.data_ptr<int>(), (int)nt, (int)B, (int)d.H, (int)d.D,
      (int)d.E, st, (float)qscale, (float)eps, stream());
}

void recurrent_out(torch::Tensor y, torch::Tensor o, torch::Tensor g,
                   torch::Tensor w, long heads, bool mlstm, double eps) {
  const auto dt = y.scalar_type();
  const long rows = g.size(0), HE = g.size(1), E = HE / heads;
  TORCH_CHECK(HE % heads == 0, "recurrent_out: heads");
  check(y, dt, "y");
  TORCH_CHECK(y.numel() == rows * HE, "recurrent_out: y");
  check_param(o, rows * HE, "o");
  check_rows(g, dt, rows, HE, g.stride(0), "g");
  check_param(w, mlstm ? HE : E, "norm weight");
  by_dtype(y, [&](auto tag) {
    using T = ELEM(tag);
    launch_recurrent_out<T>(ptr<T>(y), ptr<float>(o), ptr<T>(g),
                            ptr<float>(w), mlstm, rows, (int)heads, (int)E,
                            g.stride(0), (float)eps, stream());
  });
}

void check_step(const torch::Tensor& y, const StateDims& d,
                const torch::Tensor& q, const torch::Tensor& k,
                const torch::Tensor& v, const torch::Tensor& g,
                const torch::Tensor& positions, const torch::Tensor& slots) {
  const auto dt = q.scalar_type();
  const long rows = q.size(0), st = q.stride(0);
  check(y, dt, "y");
  TORCH_CHECK(y.numel() == rows * d.H * d.E, "recurrent_step: y");
  check_rows(q, dt, rows, d.H * d.D, st, "q");
  check_rows(k, dt, rows, d.H * d.D, st, "k");
  check_rows(v, dt, rows, d.H * d.E, st, "v");
  check_rows(g, dt, rows, d.H * d.E, st, "g");
  check(positions, torch::kInt64, "positions");
  check(slots, torch::kInt32, "slots");
  TORCH_CHECK(positions.numel() == rows && slots.numel() == rows,
              "recurrent_step: rows");
}

void gla_step(torch::Tensor y, torch::Tensor S, torch::Tensor q,
              torch::Tensor k, torch::Tensor v, torch::Tensor g,
              torch::Tensor a1h, torch::Tensor a2, torch::Tensor a2b,
              torch::Tensor w, torch::Tensor positions, torch::Tensor slots,
              double qscale, double tau, double eps) {
  const auto d = check_state(S, c10::nullopt, c10::nullopt);
  check_step(y, d, q, k, v, g, positions, slots);
  const long rows = q.size(0), R = a2.size(1);
  check_rows(a1h, q.scalar_type(), rows, R, q.stride(0), "a1h");
  check(a2, q.scalar_type(), "a2");
  TORCH_CHECK(a2.size(0) == d.H * d.D, "gla_step: a2");
  check_param(a2b, d.H * d.D, "a2 bias");
  check_param(w, d.E, "norm weight");
  by_dtype(q, [&](auto tag) {
    using T = ELEM(tag);
    launch_recurrent_step<T>(
        GLA, ptr<T>(y), nullptr, ptr<float>(S), nullptr, nullptr, ptr<T>(q),
        ptr<T>(k),
        ptr<T>(v), ptr<T>(g), ptr<T>(a1h), ptr<T>(a2), ptr<float>(a2b),
        nullptr, nullptr, ptr<float>(w), positions.data_ptr<long>(),
        slots.data_ptr<int>(), rows, (int)d.H, (int)d.D, (int)d.E, (int)R,
        q.stride(0), (float)qscale, (float)tau, (float)eps, stream());
  });
}

void mlstm_step(torch::Tensor y, torch::Tensor S, torch::Tensor n,
                torch::Tensor m, torch::Tensor q, torch::Tensor k,
                torch::Tensor v, torch::Tensor g, torch::Tensor raw,
                torch::Tensor ib, torch::Tensor fb, torch::Tensor w,
                torch::Tensor positions, torch::Tensor slots, double qscale,
                double cap, double eps) {
  const auto d = check_state(S, n, m);
  check_step(y, d, q, k, v, g, positions, slots);
  const long rows = q.size(0);
  check_param(raw, rows * 2 * d.H, "raw gates");
  check_param(ib, d.H, "input gate bias");
  check_param(fb, d.H, "forget gate bias");
  check_param(w, d.H * d.E, "norm weight");
  by_dtype(q, [&](auto tag) {
    using T = ELEM(tag);
    launch_recurrent_step<T>(
        MLSTM, ptr<T>(y), nullptr, ptr<float>(S), ptr<float>(n),
        ptr<float>(m), ptr<T>(q),
        ptr<T>(k), ptr<T>(v), ptr<T>(g), nullptr, nullptr, ptr<float>(ib),
        ptr<float>(fb), ptr<float>(raw), ptr<float>(w),
        positions.data_ptr<long>(), slots.data_ptr<int>(), rows, (int)d.H,
        (int)d.D, (int)d.E, 0, q.stride(0), (float)qscale, (float)cap,
        (float)eps, stream());
  });
}

// q, k, v rows of one buffer, o [T, H * E] float, one decay per head
StateDims check_lightning(const torch::Tensor& o, const torch::Tensor& S,
                          const torch::Tensor& q, const torch::Tensor& k,
                          const torch::Tensor& v, const torch::Tensor& decay,
                          const torch::Tensor& positions,
                          const torch::Tensor& slots) {
  const auto d = check_state(S, c10::nullopt, c10::nullopt);
  const auto dt = q.scalar_type();
  const long rows = q.size(0), st = q.stride(0);
  check_rows(q, dt, rows, d.H * d.D, st, "q");
  check_rows(k, dt, rows, d.H * d.D, st, "k");
  check_rows(v, dt, rows, d.H * d.E, st, "v");
  check_param(o, rows * d.H * d.E, "o");
  check_param(decay, d.H, "decay");
  check(positions, torch::kInt64, "positions");
  check(slots, torch::kInt32, "slots");
  TORCH_CHECK(positions.numel() == rows, "lightning: rows");
  return d;
}

void lightning_step(torch::Tensor o, torch::Tensor S, torch::Tensor q,
                    torch::Tensor k, torch::Tensor v, torch::Tensor decay,
                    torch::Tensor positions, torch::Tensor slots) {
  const auto d = check_lightning(o, S, q, k, v, decay, positions, slots);
  TORCH_CHECK(slots.numel() == q.size(0), "lightning_step: slots");
  by_dtype(q, [&](auto tag) {
    using T = ELEM(tag);
    launch_recurrent_step<T>(
        LIGHTNING, nullptr, ptr<float>(o), ptr<float>(S), nullptr, nullptr,
        ptr<T>(q), ptr<T>(k), ptr<T>(v), nullptr, nullptr, nullptr,
        ptr<float>(decay), nullptr, nullptr, nullptr,
        positions.data_ptr<long>(), slots.data_ptr<int>(), q.size(0),
        (int)d.H, (int)d.D, (int)d.E, 0, q.stride(0), 1.f, 0.f, 0.f,
        stream());
  });
}

void lightning_scan(torch::Tensor o, torch::Tensor S, torch::Tensor q,
                    torch::Tensor k, torch::Tensor v, torch::Tensor decay,
                    torch::Tensor seq_start, torch::Tensor positions,
                    torch::Tensor slots) {
  const auto d = check_lightning(o, S, q, k, v, decay, positions, slots);
  const long B = slots.numel();
  check(seq_start, torch::kInt32, "seq_start");
  TORCH_CHECK(seq_start.numel() == B + 1 && B <= 65535,
              "lightning_scan: sequences");
  by_dtype(q, [&](auto tag) {
    using T = ELEM(tag);
    launch_recurrent_scan<T>(
        LIGHTNING, ptr<float>(o), ptr<float>(S), nullptr, nullptr, nullptr,
        ptr<T>(q), ptr<T>(k), ptr<T>(v), ptr<float>(decay),
        seq_start.data_ptr<int>(), positions.data_ptr<long>(),
        slots.data_ptr<int>(), (int)B, (int)d.H, (int)d.D, (int)d.E,
        q.stride(0), 1.f, stream());
  });
}

void lightning_chunk(torch::Tensor o, torch::Tensor U, torch::Tensor S,
                     torch::Tensor q, torch::Tensor k, torch::Tensor v,
                     torch::Tensor decay, torch::Tensor seq_start,
                     torch::Tensor positions, torch::Tensor slots,
                     torch::Tensor tiles, torch::Tensor tile_start) {
  const auto d = check_lightning(o, S, q, k, v, decay, positions, slots);
  const long B = slots.numel(), nt = tiles.size(0);
  TORCH_CHECK(chunk_fits(S, q, k, v, v, 0), "lightning_chunk: sizes");
  check(tile_start, torch::kInt32, "tile_start");
  check_tiles(tiles, seq_start, B);
  TORCH_CHECK(tile_start.numel() == B + 1 && B <= 65535,
              "lightning_chunk: sequences");
  check_param(U, nt * d.H * d.D * d.E, "U");
  launch_recurrent_chunk(
      LIGHTNING, nullptr, ptr<float>(o), ptr<float>(U), nullptr, nullptr,
      ptr<float>(S), nullptr, nullptr, ptr<bf16>(q), ptr<bf16>(k),
      ptr<bf16>(v), nullptr, ptr<float>(decay), nullptr, nullptr,
      seq_start.data_ptr<int>(), positions.data_ptr<long>(),
      slots.data_ptr<int>(), tiles.data_ptr<int>(),
      tile_start.data_ptr<int>(), (int)nt, (int)B, (int)d.H, (int)d.D,
      (int)d.E, q.stride(0), 1.f, 0.f, stream());
}

void greedy_sample(torch::Tensor out, torch::Tensor logits) {
  check(out, torch::kInt64, "out");
  if (logits.scalar_type() == torch::kFloat32) {
    check(logits, torch::kFloat32, "logits");
    launch_greedy_sample(out.data_ptr<long>(), logits.data_ptr<float>(),
                         logits.size(0), (int)logits.size(1), stream());
    return;
  }
  check(logits, torch::kBFloat16, "logits");
  launch_greedy_sample(out.data_ptr<long>(), cbf(logits), logits.size(0),
                       (int)logits.size(1), stream());
}

void sample(torch::Tensor out, torch::Tensor logits,
            torch::Tensor temperature, torch::Tensor top_p,
            torch::Tensor top_k, torch::Tensor uniform) {
  check(out, torch::kLong, "out");
  check(logits, logits.scalar_type(), "logits");
  TORCH_CHECK(logits.dim() == 2 && logits.size(1) > 0 &&
                  logits.size(1) < (1l << 23), "logits");
  const long rows = logits.size(0);
  TORCH_CHECK(out.numel() == rows, "out");
  check_param(temperature, rows, "temperature");
  check_param(top_p, rows, "top_p");
  check(top_k, torch::kInt32, "top_k");
  TORCH_CHECK(top_k.numel() == rows, "top_k");
  check_param(uniform, rows, "uniform");
  const long bytes = sample_workspace(rows, (int)logits.size(1));
  torch::Tensor ws;
  if (bytes) ws = torch::empty({bytes}, out.options().dtype(torch::kUInt8));
  by_dtype(logits, [&](auto tag) {
    using T = ELEM(tag);
    launch_sample<T>(out.data_ptr<long>(), ptr<T>(logits),
                     ptr<float>(temperature), ptr<float>(top_p),
                     top_k.data_ptr<int>(), ptr<float>(uniform),
                     bytes ? ws.data_ptr() : nullptr, rows,
                     (int)logits.size(1), stream());
  });
}

}  // namespace


unsigned char* u8(torch::Tensor& t) {
  return reinterpret_cast<unsigned char*>(t.data_ptr());
}

void quant_fp8(torch::Tensor out, torch::Tensor scales, torch::Tensor x) {
  check(out, torch::kFloat8_e4m3fn, "out");
  check(scales, torch::kFloat, "scales");
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == torch::kBFloat16, "x");
  const int hidden = (int)x.size(-1);
  TORCH_CHECK(x.stride(-1) == 1, "x inner dim must be contiguous");
  const long rows = x.numel() / hidden;
  const long stride = x.dim() > 1 ? x.stride(0) : hidden;
  launch_quant_fp8(u8(out), scales.data_ptr<float>(), cbf(x), rows, hidden,
                   stride, stream());
}

void fused_add_rmsnorm_fp8(torch::Tensor out, torch::Tensor scales,
                           torch::Tensor x, torch::Tensor residual,
                           torch::Tensor w, double eps) {
  check(out, torch::kFloat8_e4m3fn, "out");
  check(scales, torch::kFloat, "scales");
  check(x, torch::kBFloat16, "x");
  check(residual, torch::kBFloat16, "residual");
  check(w, torch::kBFloat16, "w");
  const int hidden = (int)x.size(-1);
  launch_fused_add_rmsnorm_fp8(u8(out), scales.data_ptr<float>(), cbf(x),
                               bf(residual), cbf(w), (float)eps,
                               x.numel() / hidden, hidden, stream());
}

// the same, x the sum of float parts [parts, rows, hidden]
void parts_add_rmsnorm_fp8(torch::Tensor out, torch::Tensor scales,
                           torch::Tensor parts, torch::Tensor residual,
                           torch::Tensor w, double eps) {
  check(out, torch::kFloat8_e4m3fn, "out");
  check(scales, torch::kFloat, "scales");
  check(parts, torch::kFloat, "parts");
  check(residual, torch::kBFloat16, "residual");
  check(w, torch::kBFloat16, "w");
  TORCH_CHECK(parts.dim() == 3 && parts.size(0) >= 2 && parts.size(0) <= 8,
              "parts_add_rmsnorm_fp8: 2 to 8 parts");
  const long rows = parts.size(1);
  const int hidden = (int)parts.size(2);
  TORCH_CHECK(hidden % 8 == 0 && hidden <= 8192 && w.numel() == hidden &&
                  out.numel() == rows * hidden && scales.numel() == rows &&
                  residual.numel() == out.numel(),
              "parts_add_rmsnorm_fp8: shape");
  if (rows == 0) return;
  launch_parts_add_rmsnorm_fp8(
      u8(out), scales.data_ptr<float>(), parts.data_ptr<float>(),
      (int)parts.size(0), bf(residual), cbf(w), (float)eps, rows, hidden,
      stream());
}

void silu_mul_fp8(torch::Tensor out, torch::Tensor scales, torch::Tensor x) {
  check(out, torch::kFloat8_e4m3fn, "out");
  check(scales, torch::kFloat, "scales");
  check(x, torch::kBFloat16, "x");
  const int inter = (int)out.size(-1);
  TORCH_CHECK(x.size(-1) == 2 * inter, "x must be [rows, 2*inter]");
  launch_silu_mul_fp8(u8(out), scales.data_ptr<float>(), cbf(x),
                      out.numel() / inter, inter, stream());
}


void moe_gemm(torch::Tensor out, torch::Tensor x, torch::Tensor w,
              torch::Tensor sorted_ids, torch::Tensor tile_expert,
              long gather_div, long splitk,
              c10::optional<torch::Tensor> ws) {
  check(out, torch::kBFloat16, "out");
  check(x, torch::kBFloat16, "x");
  check(w, torch::kBFloat16, "w");
  check(sorted_ids, torch::kInt, "sorted_ids");
  check(tile_expert, torch::kInt, "tile_expert");
  TORCH_CHECK(w.dim() == 3, "w must be [E, N, K]");
  float* wsp = nullptr;
  if (splitk > 1) {
    TORCH_CHECK(ws.has_value(), "moe_gemm: splitk>1 needs a workspace");
    check(*ws, torch::kFloat, "ws");
    TORCH_CHECK(ws->numel() >= splitk * out.numel(),
                "moe_gemm: workspace too small");
    wsp = ws->data_ptr<float>();
  }
  launch_moe_gemm(bf(out), wsp, cbf(x), cbf(w),
                  sorted_ids.data_ptr<int>(),
                  tile_expert.data_ptr<int>(), (int)tile_expert.numel(),
                  (int)w.size(1), (int)w.size(2), (int)gather_div,
                  (int)splitk, stream());
}


void register_latent(pybind11::module_& m);    // bindings_latent.cpp
void register_sublayer(pybind11::module_& m);  // bindings_sublayer.cpp

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "HyperSpot-AMD gfx950 (CDNA4) kernels";
  m.def("rmsnorm", &rmsnorm);
  m.def("quant_fp8", &quant_fp8);
  m.def("fused_add_rmsnorm_fp8", &fused_add_rmsnorm_fp8);
  m.def("parts_add_rmsnorm_fp8", &parts_add_rmsnorm_fp8);
  m.def("silu_mul_fp8", &silu_mul_fp8);
  m.def("gemm_wide", &gemm_wide, py::arg("out"), py::arg("x"), py::arg("w"),
        py::arg("part"), py::arg("high"), py::arg("bn"), py::arg("splits") = 1,
        py::arg("gated") = false);
  m.def("moe_gemm", &moe_gemm);
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm);
  m.def("rope_kv_append", &rope_kv_append);
  m.def("paged_attn", &paged_attn);
  m.def("rope_paged_attn", &rope_paged_attn);
  m.def("attn_prefill_mfma", &attn_prefill_mfma);
  m.def("attn_portions", &attn_portions);
  m.def("decode_inputs", &decode_inputs);
  m.def("gemm_rows", &gemm_rows, pybind11::arg("out"), pybind11::arg("x"),
        pybind11::arg("w"), pybind11::arg("x_scale") = pybind11::none(),
        pybind11::arg("w_scale") = pybind11::none());
  m.def("gemm_rows_fits", &gemm_rows_fits);
  m.def("gemm_split", &gemm_split, pybind11::arg("out"), pybind11::arg("x"),
        pybind11::arg("w"), pybind11::arg("part"), pybind11::arg("bm"),
        pybind11::arg("bn"), pybind11::arg("splits"),
        pybind11::arg("x_scale") = pybind11::none(),
        pybind11::arg("w_scale") = pybind11::none(),
        pybind11::arg("gated") = false);
  m.def("parts_add_rmsnorm", &parts_add_rmsnorm);
  m.def("experts_few", &experts_few);
  m.def("choices_add_rmsnorm", &choices_add_rmsnorm);
  m.def("silu_mul", &silu_mul);
  m.def("gelu_mul", &gelu_mul);
  m.def("embed_dyt", &embed_dyt);
  m.def("add_dyt", &add_dyt);
  m.def("rope_pairs_append", &rope_pairs_append);
  m.def("window_attn_general", &window_attn_general);
  m.def("window_attn_fits", &window_attn_fits);
  m.def("window_attn_prefill", &window_attn_prefill);
  m.def("window_attn_decode", &window_attn_decode);
  m.def("gla_chunk_gates", &gla_chunk_gates);
  m.def("mlstm_chunk_gates", &mlstm_chunk_gates);
  m.def("chunk_fits", &chunk_fits);
  m.def("recurrent_chunk", &recurrent_chunk);
  m.def("gla_decay", &gla_decay);
  m.def("mlstm_gates", &mlstm_gates);
  m.def("recurrent_scan", &recurrent_scan);
  m.def("recurrent_out", &recurrent_out);
  m.def("gla_step", &gla_step);
  m.def("mlstm_step", &mlstm_step);
  m.def("lightning_step", &lightning_step);
  m.def("lightning_scan", &lightning_scan);
  m.def("lightning_chunk", &lightning_chunk);
  register_latent(m);
  register_sublayer(m);
  m.def("greedy_sample", &greedy_sample);
  m.def("sample", &sample);
}
