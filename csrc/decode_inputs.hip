// The inputs of a captured decode step from one staged copy (gfx950).
//
// The host stages five values a row and the rows' page ids in one buffer; this
// kernel puts them where the graph reads them, pads the rows up to the graph's
// batch and clears the rest of the page table.  What bounds it is the launch:
// it replaces five copies and ten fills and slice copies, 2 to 4 us each on a
// step's critical path.
#include "common.h"

namespace {

struct DecodeInputs {
  const long* stage;         // [5, cap]: id, position, slot, tokens, state row
  const int* pages;          // [B, staged]
  long* ids;                 // [bucket] each
  long* positions;
  long* slots;
  int* lens;
  int* state;                // null: none
  int* tables;               // [bucket, max_blocks]
  int B, bucket, cap, staged, max_blocks;
};

__global__ __launch_bounds__(256) void decode_inputs_kernel(DecodeInputs a) {
  const int r = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  const bool row = r < a.B;
  if (c < a.max_blocks)
    a.tables[(long)r * a.max_blocks + c] =
        row && c < a.staged ? a.pages[(long)r * a.staged + c] : 0;
  if (c) return;
  // padding: a row of one token that writes nothing
  const long* s = a.stage + r;
  a.ids[r] = row ? s[0] : 0;
  a.positions[r] = row ? s[a.cap] : 0;
  a.slots[r] = row ? s[2l * a.cap] : -1;
  a.lens[r] = row ? (int)s[3l * a.cap] : 1;
  if (a.state) a.state[r] = row ? (int)s[4l * a.cap] : -1;
}

}  // namespace

void launch_decode_inputs(const long* stage, const int* pages, long* ids,
                          long* positions, long* slots, int* lens, int* state,
                          int* tables, int B, int bucket, int cap, int staged,
                          int max_blocks, hipStream_t stream) {
  if (bucket == 0) return;
  decode_inputs_kernel<<<dim3((unsigned)bucket,
                              (unsigned)((max_blocks + 255) / 256)),
                         256, 0, stream>>>(
      {stage, pages, ids, positions, slots, lens, state, tables, B, bucket,
       cap, staged, max_blocks});
}
