// Sampling kernels: greedy argmax, and the whole of temperature, top-k, top-p
// and draw.
//
// A batch row of vocab-size logits (128256 for Llama-3) is one workgroup's, or
// that of several and a second kernel where there are few rows.  Vectorized
// bf16/f32 reads; fp32 math, sums of weights in 64-bit integers.
#include <float.h>

#include <type_traits>

#include "common.h"

// ---- greedy argmax (bf16 or float logits) ------------------------------
template <typename T>
__global__ __launch_bounds__(256) void greedy_sample_kernel(
    long* __restrict__ out, const T* __restrict__ logits, int vocab) {
  __shared__ float smax[4];
  __shared__ int sidx[4];
  const T* row = logits + (long)blockIdx.x * vocab;
  float best = -FLT_MAX;
  int besti = 0;
  int done = 0;                        // elements covered by the vector part
  if constexpr (sizeof(T) == 2) {
    // rows start 16-byte aligned only when the vocabulary is a multiple of 8
    if (vocab % 8 == 0) {
      done = vocab;
      for (int u = threadIdx.x; u < vocab / 8; u += 256) {
        bf16x8 v = load_bf16x8(row + u * 8);
        #pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float f = bf16x8_get(v, i);
          if (f > best) { best = f; besti = u * 8 + i; }
        }
      }
    }
  }
  for (int t = done + threadIdx.x; t < vocab; t += 256) {
    const float f = Elem<T>::ld(row + t);
    if (f > best) { best = f; besti = t; }
  }
  // wave reduce (value, index) — ties resolve to the smaller index like
  // torch.argmax on contiguous fp32
  #pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o);
    const int oi = __shfl_xor(besti, o);
    if (ob > best || (ob == best && oi < besti)) { best = ob; besti = oi; }
  }
  const int wid = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { smax[wid] = best; sidx[wid] = besti; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w)
      if (smax[w] > best || (smax[w] == best && sidx[w] < besti)) {
        best = smax[w]; besti = sidx[w];
      }
    out[blockIdx.x] = besti;
  }
}

// ---- temperature, top-k, top-p and draw ---------------------------------
// Row b: weights exp(x / max(temperature, 1e-6)) of the logits x; with 0 <
// top_k < vocab the values below the top_k-th largest go (its equals stay);
// with top_p < 1 a token goes if the ones before it, in descending order and
// by index among equals, have at least top_p of the weight; the first token
// at which the running sum of the others exceeds uniform * sum is drawn.
// temperature 0: the largest logit, the first among equals.  A logit that is
// NaN is not drawn.
//
// What bounds it: vector instructions on every value, 14 (the exponential as 4) for
// a weight of less than 2^-12 of the largest and 19 for another, and the chains of
// steps that a row's workgroup takes one after the other.  So a row is divided into
// slices where there are few rows (below): 64 rows of 128256 are 256 workgroups,
// which have the largest values after 2.5 us and the weights after 6; a second kernel
// of a workgroup a row takes 2 (greedy) to 4.5 us (a share).  Lanes are combined by
// DPP, and what the 16 waves found by 16 lanes: with shuffles, and with every lane
// adding up 16 values, a mix of options took 24.3 us, so 21.9.  8 values are looked at
// together where that decides about all of them.
// Where few values stay, and next-token logits have a few dozen that matter, they
// are listed and the rest is done on the list, up to 8 threads a value.  n values
// take n^2 steps, so the lists are kept short.  Each slice lists its own largest, so
// many that a share is found among the 64 largest of the row, or top_k up to 100:
// that takes 0.8 us where weights are computed and 2 where not, and the second kernel
// has the row's list without a pass of its own over the row, which took it 4.5 us (a
// mix 19.0 -> 14.5 us with the sums of weights, below).  Where that list is too short,
// the second kernel makes one of 128 (or of top_k up to 256), as before.
// Otherwise no sort either: one histogram of counts and weights over 2048 equal steps
// between the largest and the smallest logit finds the step where the wanted count or
// share is reached, and ranks the few values in it exactly (or divides that step
// again).  Equal steps of the logit, and not digits of its bit pattern, because
// next-token logits fill few exponents: 64 lanes that add to the same few counters in
// LDS would go one by one.
//
// 64 rows of 128256 in bfloat16, 48 values far above the others, us with a workgroup
// a row, in slices, and with lists of the slices (rows in cache; from memory 2 to 3
// more): temperature 36 14.1 12.5, top_p 0.9 43 20.2 15.6, top_k 50 24 13.7 12.6,
// greedy 9.4 7.8 7.9; a mix 42 19.9 15.6, where the library's sorts, scans and
// selections took 2625.  A mix of 1 row 16.4 -> 13.4, of 128 27.2 -> 24.0; 64 rows of
// 32000 17.2 -> 13.9.  What the lists cost where they do not help: top_k of 65 to 128
// rows of 128256, which are two workgroups a compute unit, 2 to 4 % (50 of 128 17.6 ->
// 18.0; without them a mix loses, 24.0 -> 26.5), greedy rows if they are few 0.3 (16 7.4
// -> 7.8).  A call that is waited for and not captured 60 36.
//
// Weights are 2^-40 fixed point relative to the largest (of the row or of the
// slice), so sums within a row or a slice are exact; slices are brought to the
// row's scale by one rounded factor each and added in their order.  So the same
// inputs give the same token; a batch of another size, which is divided
// otherwise, may give another one where the draw falls on a boundary to 2^-40.
namespace {

typedef unsigned long long u64;
constexpr int NT = 1024;          // threads
constexpr int STEPS = 2048;       // of the histogram
constexpr int LIST = 512;         // values ranked one by one
constexpr int AHEAD = 2;          // loads of a thread on their way
constexpr int FEW = 128;          // values that a share is looked for in

struct Weight {
  float mx, hi, lo;               // hi + lo = log2(e) / temperature
  // to be cut to a whole number
  DEV float scaled(float x) const {
    const float d = x - mx, t = d * hi;
    const float r = fmaf(d, hi, -t) + d * lo;
    const float e = __builtin_amdgcn_exp2f(t);
    return fmaf(e * r, 0.69314718f, e) * 1099511627776.f + 0.5f;
  }
  // false: weights of x and less are below half of 2^-40
  DEV bool any(float x) const { return (x - mx) * hi > -42.f; }
  DEV u64 operator()(float x) const { return any(x) ? always(x) : 0; }
  // the same of less than 2^-8 of the largest; 8 of less than 2^-12 add up to 32 bits
  DEV unsigned small(float x) const {
    return (unsigned)scaled(x);
  }
  // the same without a branch: the weights that `any` rules out, an infinity's
  // and a NaN's among them, come out as zero
  DEV u64 always(float x) const {
    const float e = scaled(x);
    const unsigned h = (unsigned)(e * 2.3283064e-10f);
    return (u64)h << 32 | (unsigned)fmaf((float)h, -4294967296.f, e);
  }
};

// order-preserving bits
DEV unsigned ordered(float x) {
  const unsigned u = __float_as_uint(x);
  return u & 0x80000000u ? ~u : u | 0x80000000u;
}
DEV float from_ordered(unsigned u) {
  return __uint_as_float(u & 0x80000000u ? u & 0x7fffffffu : ~u);
}

// an infinity as the largest finite value; NaN, which is never drawn, as -inf
DEV float in_range(float x) { return fminf(fmaxf(x, -INFINITY), FLT_MAX); }

DEV float largest(const float* x) {
  return fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])),
               fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
}
DEV float smallest(const float* x) {
  return fminf(fminf(fminf(x[0], x[1]), fminf(x[2], x[3])),
               fminf(fminf(x[4], x[5]), fminf(x[6], x[7])));
}

// Combinations over lanes by DPP, which takes a few cycles a step where a shuffle
// goes through LDS.  x of another lane, or `none` where CTRL and the rows of
// ROWS have no such lane:
template <int CTRL, int ROWS, typename I> DEV I from_lane(I x, I none) {
  if constexpr (sizeof(I) == 8) {
    const u64 a = __builtin_bit_cast(u64, x), b = __builtin_bit_cast(u64, none);
    const u64 lo = from_lane<CTRL, ROWS>((unsigned)a, (unsigned)b);
    const u64 hi = from_lane<CTRL, ROWS>((unsigned)(a >> 32),
                                         (unsigned)(b >> 32));
    return __builtin_bit_cast(I, hi << 32 | lo);
  } else {
    return __builtin_bit_cast(I, __builtin_amdgcn_update_dpp(
        __builtin_bit_cast(int, none), __builtin_bit_cast(int, x), CTRL, ROWS,
        0xf, false));
  }
}
// f over the lanes of 16 up to this one: row_shr by 1, 2, 4 and 8
template <typename I, typename F> DEV I row_scan(I x, I none, F f) {
  x = f(x, from_lane<0x111, 0xf>(x, none));
  x = f(x, from_lane<0x112, 0xf>(x, none));
  x = f(x, from_lane<0x114, 0xf>(x, none));
  return f(x, from_lane<0x118, 0xf>(x, none));
}
// f over the lanes up to this one, then row_bcast of lanes 15 and 31
template <typename I, typename F> DEV I wave_scan(I x, I none, F f) {
  x = row_scan(x, none, f);
  x = f(x, from_lane<0x142, 0xa>(x, none));
  return f(x, from_lane<0x143, 0xc>(x, none));
}
template <typename I> DEV I wave_scan(I x) {      // inclusive sums
  return wave_scan(x, I(0), [](I a, I b) { return a + b; });
}
// x[i % 4] summed over the lanes, in lane i: one step divides the four among
// two neighbours, the next among four
DEV u64 wave_sums(const u64* x) {
  const int lane = threadIdx.x;
  const bool odd = lane & 1, high = lane & 2;
  const u64 a = (odd ? x[1] : x[0]) +
                from_lane<0xb1, 0xf>(odd ? x[0] : x[1], u64(0));
  const u64 b = (odd ? x[3] : x[2]) +
                from_lane<0xb1, 0xf>(odd ? x[2] : x[3], u64(0));
  u64 c = (high ? b : a) + from_lane<0x4e, 0xf>(high ? a : b, u64(0));
  c += from_lane<0x124, 0xf>(c, u64(0));          // row_ror by 4 and 8
  c += from_lane<0x128, 0xf>(c, u64(0));
  c += __shfl_xor(c, 16);
  return c + __shfl_xor(c, 32);
}
template <typename I> DEV I lane_of(I x, int lane) {       // uniform
  if constexpr (sizeof(I) == 8) {
    const u64 a = __builtin_bit_cast(u64, x);
    const u64 lo = (unsigned)__builtin_amdgcn_readlane((int)a, lane);
    const u64 hi = (unsigned)__builtin_amdgcn_readlane((int)(a >> 32), lane);
    return __builtin_bit_cast(I, hi << 32 | lo);
  } else {
    return __builtin_bit_cast(
        I, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
  }
}
// the sum of 16 values in LDS, and of those before `before` of them; all lanes
template <typename I> DEV I sum_of_16(const I* x, int before, I* sum) {
  const I upto = row_scan(x[threadIdx.x & 15], I(0),
                          [](I a, I b) { return a + b; });
  *sum = lane_of(upto, 15);
  return before ? lane_of(upto, before - 1) : I(0);
}
// the sum alone: row_ror by 8, 4, 2 and 1
DEV u64 sum_of_16(const u64* x) {
  u64 y = x[threadIdx.x & 15];
  y += from_lane<0x128, 0xf>(y, u64(0));
  y += from_lane<0x124, 0xf>(y, u64(0));
  y += from_lane<0x122, 0xf>(y, u64(0));
  return y + from_lane<0x121, 0xf>(y, u64(0));
}
DEV float min_of(float a, float b) { return fminf(a, b); }

struct alignas(16) Entry {        // one LDS load
  u64 key, mass;
};

struct Scratch {
  u64 mass[STEPS];
  unsigned count[STEPS];
  float list[LIST];
  int list_at[LIST];
  Entry entry[LIST];
  u64 wave_mass[16];
  unsigned wave_count[16];
  u64 before_mass, kept_mass, list_mass[16];
  unsigned before_count, n, key_min, key_max, keep, stay;
  int step, found;
  float value;
};

// VEC: 8 elements of a row at a time, 16-byte aligned
template <typename T, bool VEC> struct Row {
  const T* p;
  int vocab;
  bool finite;                    // no value is above FLT_MAX, or it may be
  typedef __attribute__((ext_vector_type(8))) float f32x8;
  struct Raw {                    // as loaded: nothing waits for it yet
    typename std::conditional<sizeof(T) == 2, uint4, f32x8>::type v;
  };
  // the elements [at, at + 8), -inf from `end` on; not above FLT_MAX unless
  // `finite` says so
  DEV void fetch(int at, int end, Raw& r) const {
    if constexpr (VEC) {
      if (at < end)
        r.v = *reinterpret_cast<const decltype(r.v)*>(p + at);
      else if constexpr (sizeof(T) == 2)
        r.v = uint4{0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
      else
        r.v = f32x8(-INFINITY);
    }
  }
  DEV void unpack(const Raw& r, int at, int end, float* x) const {
    if constexpr (!VEC) {
      #pragma unroll
      for (int i = 0; i < 8; ++i)
        x[i] = at + i < end ? Elem<T>::ld(p + at + i) : -INFINITY;
    } else if constexpr (sizeof(T) == 2) {
      const unsigned u[4] = {r.v.x, r.v.y, r.v.z, r.v.w};
      #pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[2 * i] = __uint_as_float(u[i] << 16);
        x[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
      }
    } else {
      #pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = r.v[i];
    }
    if (!finite)
      #pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = in_range(x[i]);
  }
  // the same from anywhere: elements one by one where they are not aligned
  DEV void hold(int at, int end, Raw& r) const {
    if constexpr (VEC) {
      fetch(at, end, r);
    } else if constexpr (sizeof(T) == 2) {
      unsigned u[4];
      #pragma unroll
      for (int i = 0; i < 4; ++i) {
        unsigned h[2];
        #pragma unroll
        for (int j = 0; j < 2; ++j)
          h[j] = at + 2 * i + j < end
              ? reinterpret_cast<const unsigned short*>(p)[at + 2 * i + j]
              : 0xff80u;
        u[i] = h[0] | h[1] << 16;
      }
      r.v = uint4{u[0], u[1], u[2], u[3]};
    } else {
      #pragma unroll
      for (int i = 0; i < 8; ++i)
        r.v[i] = at + i < end ? Elem<T>::ld(p + at + i) : -INFINITY;
    }
  }
  DEV void spread(const Raw& r, float* x) const {
    Row<T, true>{p, vocab, finite}.unpack({r.v}, 0, 0, x);
  }
  // f(8 values, index of the first) of all values and of some -inf past the end
  template <typename F> DEV void each8(F f) const {
    for (int at = threadIdx.x * 8; at < vocab; at += AHEAD * NT * 8) {
      Raw r[AHEAD];
      #pragma unroll
      for (int q = 0; q < AHEAD; ++q) fetch(at + q * NT * 8, vocab, r[q]);
      #pragma unroll
      for (int q = 0; q < AHEAD; ++q) {
        float x[8];
        unpack(r[q], at + q * NT * 8, vocab, x);
        f(x, at + q * NT * 8);
      }
    }
  }
  template <typename F> DEV void each(F f) const {
    each8([&](const float* x, int at) {
      #pragma unroll
      for (int i = 0; i < 8; ++i) f(x[i], at + i);
    });
  }

  // First index in [first, end) at which the running sum of w(x, index) exceeds
  // the target that `of` makes of the whole sum; vocab - 1 if there is none.  A
  // wave has a sixteenth; the one where the target lies is divided again.
  template <typename W, typename F>
  DEV int walk(Scratch& s, W w, F of, int first, int end) const {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    u64 before = 0, target = 0;
    for (bool whole = true;; whole = false) {
      const int span = (end - first + 16 * 512 - 1) / (16 * 512) * 512;
      const int mine = first + wid * span, stop = min(mine + span, end);
      float x[8];                 // the first ones
      u64 sum = 0;
      for (int at = mine + lane * 8; at < stop; at += AHEAD * 512) {
        Raw r[AHEAD];
        #pragma unroll
        for (int q = 0; q < AHEAD; ++q) fetch(at + q * 512, stop, r[q]);
        #pragma unroll
        for (int q = AHEAD - 1; q >= 0; --q) {
          unpack(r[q], at + q * 512, stop, x);
          #pragma unroll
          for (int i = 0; i < 8; ++i) sum += w(x[i], at + q * 512 + i);
        }
      }
      const u64 upto = wave_scan(sum);
      if (lane == 63) s.wave_mass[wid] = upto;
      __syncthreads();
      if (whole) {
        u64 total = 0;
        for (int v = 0; v < 16; ++v) total += s.wave_mass[v];
        target = of(total);
      }
      int owner = 0;
      while (owner < 16 && before + s.wave_mass[owner] <= target)
        before += s.wave_mass[owner++];
      if (owner == 16) {
        __syncthreads();
        return vocab - 1;
      }
      if (span == 512) {          // x has all of this wave's
        const u64 over = __ballot(before + upto > target);
        if (wid == owner && lane == __ffsll(over) - 1) {
          u64 c = before + upto - sum;
          for (int i = 0; i < 8; ++i)
            if ((c += w(x[i], mine + lane * 8 + i)) > target) {
              s.found = mine + lane * 8 + i;
              break;
            }
        }
        __syncthreads();
        const int found = s.found;
        __syncthreads();
        return found;
      }
      __syncthreads();
      first += owner * span;
      end = min(first + span, end);
    }
  }
  template <typename W, typename F>
  DEV int walk(Scratch& s, W w, F of) const {
    return walk(s, w, of, 0, vocab);
  }
};

// In descending order, the group of equal values in which the count reaches
// `want` (COUNT) or the weight does: s.value, s.keep of its members with less
// than `want` before them, and s.kept_mass of all values down to it.
template <bool COUNT, typename R>
DEV void reach(Scratch& s, const R& row, const Weight& w, float lo, float hi,
               u64 want) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  u64 mass0 = 0;                  // of the values above hi
  unsigned count0 = 0;
  for (int level = 0;; ++level) {
    // halves: the difference of two floats may overflow
    const float unit = STEPS / (hi * .5f - lo * .5f);
    auto step_of = [&](float x) {
      return (int)fmaxf(fminf((hi * .5f - x * .5f) * unit, STEPS - 1), 0.f);
    };
    // level 0 has all values, those below lo in the last step
    auto in = [&](float x) {
      return x <= hi && (x >= lo || (level == 0 && x >= -FLT_MAX));
    };
    for (int i = tid; i < STEPS; i += NT) s.mass[i] = s.count[i] = 0;
    __syncthreads();
    row.each([&](float x, int) {
      if (in(x)) {
        const int b = step_of(x);
        atomicAdd(&s.count[b], 1u);
        if (const u64 m = w(x)) atomicAdd(&s.mass[b], m);
      }
    });
    __syncthreads();
    // the step: two steps a thread
    {
      const int b = tid * 2;
      const u64 m = s.mass[b] + s.mass[b + 1];
      const unsigned c = s.count[b] + s.count[b + 1];
      const u64 ms = wave_scan(m);
      const unsigned cs = wave_scan(c);
      if (lane == 63) {
        s.wave_mass[wid] = ms;
        s.wave_count[wid] = cs;
      }
      if (tid == 0) {
        s.step = -1;
        s.n = 0;
        s.key_min = ~0u;
        s.key_max = 0;
      }
      __syncthreads();
      u64 mb = mass0 + ms - m;
      unsigned cb = count0 + cs - c;
      for (int v = 0; v < wid; ++v) {
        mb += s.wave_mass[v];
        cb += s.wave_count[v];
      }
      #pragma unroll
      for (int i = 0; i < 2; ++i) {
        const u64 m1 = s.mass[b + i];
        const unsigned c1 = s.count[b + i];
        if (COUNT ? cb < want && cb + c1 >= want
                  : mb < want && mb + m1 >= want) {
          s.step = b + i;
          s.before_mass = mb;
          s.before_count = cb;
        }
        mb += m1;
        cb += c1;
      }
      __syncthreads();
    }
    const int step = s.step;
    if (step < 0) {               // never reached: all values stay
      __syncthreads();
      if (tid == 0) {
        s.value = -INFINITY;
        s.keep = ~0u;
      }
      __syncthreads();
      return;
    }
    const unsigned members = s.count[step];
    mass0 = s.before_mass;
    count0 = s.before_count;
    row.each([&](float x, int) {
      if (in(x) && step_of(x) == step) {
        const unsigned at = atomicAdd(&s.n, 1u);
        if (at < LIST) {
          s.list[at] = x;
          s.entry[at].mass = w(x);
        }
        const unsigned key = ordered(x);
        if (key < s.key_min) atomicMin(&s.key_min, key);
        if (key > s.key_max) atomicMax(&s.key_max, key);
      }
    });
    __syncthreads();
    lo = from_ordered(s.key_min);
    hi = from_ordered(s.key_max);
    if (lo == hi || level == 16) {                // one group
      __syncthreads();
      if (tid == 0) {
        const u64 one = w(lo);
        s.value = lo;
        s.kept_mass = mass0 + one * members;
        s.keep = COUNT || !one ? members
                               : (unsigned)((want - mass0 + one - 1) / one);
      }
      __syncthreads();
      return;
    }
    if (members <= LIST) {
      if (tid < members) {
        const float x = s.list[tid];
        const u64 one = s.entry[tid].mass;
        u64 mb = mass0;
        unsigned cb = count0, equal = 0;
        for (unsigned j = 0; j < members; ++j) {
          const float y = s.list[j];
          equal += y == x;
          if (y > x) {
            mb += s.entry[j].mass;
            ++cb;
          }
        }
        // every member of the group writes the same
        if (COUNT ? cb < want && cb + equal >= want
                  : mb < want && mb + one * equal >= want) {
          s.value = x;
          s.kept_mass = mb + one * equal;
          s.keep = COUNT ? equal : (unsigned)((want - mb + one - 1) / one);
        }
      }
      __syncthreads();
      return;
    }
    __syncthreads();
  }
}

DEV u64 sum_of_all(Scratch& s, u64 x) {
  x = wave_scan(x);
  if ((threadIdx.x & 63) == 63) s.wave_mass[threadIdx.x >> 6] = x;
  __syncthreads();
  sum_of_16(s.wave_mass, 0, &x);
  return x;
}

// the sum over `share` neighbouring lanes: quad_perm, and row_half_mirror
template <typename I> DEV I sum_of_neighbours(I x, int share) {
  x += from_lane<0xb1, 0xf>(x, I(0));
  if (share > 2) x += from_lane<0x4e, 0xf>(x, I(0));
  if (share > 4) x += from_lane<0x141, 0xf>(x, I(0));
  return x;
}

// of the weight z; some value has it
DEV u64 part_of(float p, u64 z) { return (u64)ceil((double)p * (double)z); }

// in descending order, and by index among equals, larger keys are earlier; the
// zeros are equal
DEV u64 key_of(float x, int at) {
  return (u64)ordered(x + 0.f) << 32 | (unsigned)~at;
}

// threads a value, each with a part of the others
DEV int share_of(int n) { return n <= NT / 8 ? 8 : n <= NT / 4 ? 4 : 2; }

// Draws from the n entries, among which is all that stays, and writes the token.
// k 0: no top_k, and the first values with `part` of the weight stay.  s.stay is
// 0.
DEV void draw_from_entries(Scratch& s, int n, int vocab, int k, float p,
                           float u, u64 part, long* out) {
  const int tid = threadIdx.x;
  Entry* const stay = reinterpret_cast<Entry*>(s.mass);
  {
    const int share = share_of(n), mine = tid / share, first = tid % share;
    const bool one_of = mine < n;
    Entry own{0, 0};
    if (one_of) own = s.entry[mine];
    const unsigned value = own.key >> 32;
    int greater = 0;
    bool stays = one_of;
    if (p < 1.f) {
      u64 above = 0;
      if (one_of)
        #pragma unroll 4
        for (int j = first; j < n; j += share) {
          const Entry e = s.entry[j];
          above += e.key > own.key ? e.mass : 0;
          greater += (unsigned)(e.key >> 32) > value;
        }
      above = sum_of_neighbours(above, share);
      if (k) {
        stays = stays && sum_of_neighbours(greater, share) < k;
        part = part_of(p, sum_of_all(s, stays && first == 0 ? own.mass : 0));
      }
      stays = stays && above < part;
    } else {
      if (one_of)
        #pragma unroll 4
        for (int j = first; j < n; j += share)
          greater += (unsigned)(s.entry[j].key >> 32) > value;
      stays = stays && sum_of_neighbours(greater, share) < k;
    }
    if (stays && first == 0)
      stay[atomicAdd(&s.stay, 1u)] = {(u64)~(unsigned)own.key, own.mass};
    __syncthreads();
  }
  // in the order of indices
  n = (int)s.stay;
  const int share = share_of(n), mine = tid / share, first = tid % share;
  const bool one_of = mine < n;
  u64 all = 0, upto = 0;
  Entry own{0, 0};
  if (one_of) {
    own = stay[mine];
    #pragma unroll 4
    for (int j = first; j < n; j += share) {
      const Entry e = stay[j];
      all += e.mass;
      upto += (unsigned)e.key < (unsigned)own.key ? e.mass : 0;
    }
  }
  all = sum_of_neighbours(all, share);
  upto = sum_of_neighbours(upto, share);
  if (one_of && first == 0) {
    const u64 target = (u64)((double)u * (double)all);
    if (target >= all)
      *out = vocab - 1;
    else if (upto <= target && upto + own.mass > target)
      *out = (int)(unsigned)own.key;
  }
}

// The draw from the s.n values that are listed, if all that stays is among
// them.  k 0: no top_k, and z is the weight of all values, of which top_p is a
// share.  False if the list is too short for the share or too long.
DEV bool draw_from_list(Scratch& s, const Weight& w, int vocab, int k, float p,
                        float u, u64 z, long* out) {
  const int tid = threadIdx.x;
  const int n = (int)s.n;
  if (n > LIST) {
    __syncthreads();
    return false;
  }
  u64 mass = 0;
  if (tid == 0) s.stay = 0;
  if (tid < n) {
    mass = w(s.list[tid]);
    s.entry[tid] = {key_of(s.list[tid], s.list_at[tid]), mass};
  }
  // a list that is too short is left before its values are ranked
  u64 part = 0;
  if (k == 0 && p < 1.f) {
    part = part_of(p, z);
    if (sum_of_all(s, mass) < part) {            // a barrier on the way
      __syncthreads();
      return false;
    }
  } else {
    __syncthreads();
  }
  draw_from_entries(s, n, vocab, k, p, u, part, out);
  return true;
}

// The draw where all that stays is among few values: the want-th largest of the
// threads' own largest values has at least that many values at or above it, and
// hardly more.  Those are listed in one pass, ranked, and the token is drawn
// from the list.  k 0: no top_k, and `all` is the weight of all values.  False
// if the list is too short for the share or too long.
template <typename R>
DEV bool draw_from_few(Scratch& s, const R& row, const Weight& w, float own,
                       int k, float p, float u, u64* all, long* out) {
  const int tid = threadIdx.x;
  const int want_n = k > 0 ? k : FEW;
  const unsigned key = ordered(own);
  unsigned prefix = 0;            // 16 bits are close enough
  for (int bit = 31; bit >= 16; --bit) {
    const unsigned next = prefix | 1u << bit;
    if (__syncthreads_count(key >= next) >= want_n) prefix = next;
  }
  const float least =
      prefix > ordered(-FLT_MAX) ? from_ordered(prefix) : -FLT_MAX;
  if (tid == 0) s.n = 0;
  __syncthreads();
  u64 z = 0;                      // the share is one of this
  row.each8([&](const float* x, int at) {
    const float m = largest(x);
    if (k == 0 && w.any(m))
      #pragma unroll
      for (int i = 0; i < 8; ++i) z += w(x[i]);
    if (m >= least)
      #pragma unroll
      for (int i = 0; i < 8; ++i)
        if (x[i] >= least) {
          const unsigned n = atomicAdd(&s.n, 1u);
          if (n < LIST) {
            s.list[n] = x[i];
            s.list_at[n] = at + i;
          }
        }
  });
  z = sum_of_all(s, z);
  __syncthreads();                // the list's sum goes the same way
  *all = z;
  return draw_from_list(s, w, row.vocab, k, p, u, z, out);
}

// Best of all threads: the largest value mx, the lowest index `at` of the 8
// that hold it first, and the smallest value mn.
DEV void best_of_all(Scratch& s, float& mx, int& at, float& mn) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const auto larger = [](u64 a, u64 b) { return a > b ? a : b; };
  u64 key = wave_scan((u64)ordered(mx + 0.f) << 32 | (unsigned)~at, u64(0), larger);
  mn = wave_scan(mn, INFINITY, min_of);
  if (lane == 63) {
    s.wave_mass[wid] = key;
    s.list[wid] = mn;
  }
  __syncthreads();
  key = lane_of(row_scan(s.wave_mass[lane & 15], u64(0), larger), 15);
  mn = lane_of(row_scan(s.list[lane & 15], INFINITY, min_of), 15);
  mx = from_ordered((unsigned)(key >> 32));
  at = (int)~(unsigned)key;
  __syncthreads();
}

// The index of the largest value mx, which is among the 8 from `at` on, the
// first among equals; that of a row without a value
template <typename T>
DEV int greedy_index(const T* p, float mx, int at, int vocab, int none) {
  if (!(mx >= -FLT_MAX)) return none;
  float x[8];
  #pragma unroll
  for (int i = 0; i < 8; ++i)
    x[i] = in_range(Elem<T>::ld(p + min(at + i, vocab - 1)));
  int first = 7;
  #pragma unroll
  for (int i = 6; i >= 0; --i)
    if (x[i] == mx) first = i;
  return at + first;
}

// The draw by passes over the row.  kept: the weight of all values, or 0 where
// it is not known.
template <typename R>
DEV int draw_from_row(Scratch& s, const R& row, const Weight& w, float mn,
                      float c, int k, float p, float uniform, u64 kept) {
  const float mx = w.mx;
  // below this weights are zero
  const float floor = mx - 64.f / c;
  const float lo = mn >= -FLT_MAX ? fmaxf(mn, floor) : floor;
  float low = -INFINITY;          // values above it stay
  int last = -1;                  // and its equals up to this index
  if (k > 0) {
    reach<true>(s, row, w, lo, mx, k);
    low = s.value;
    kept = s.keep == ~0u ? 0 : s.kept_mass;
    last = row.vocab;
    __syncthreads();
  }
  if (p < 1.f) {
    if (!kept)
      row.walk(s, [&](float x, int) { return w(x); }, [&](u64 z) {
        kept = z;
        return z;
      });
    reach<false>(s, row, w, lo, mx,
                 (u64)ceil((double)p * (double)kept));
    const unsigned keep = s.keep;
    const float value = s.value;
    __syncthreads();
    if (keep != ~0u) {
      low = value;
      last = row.walk(s, [&](float x, int) { return (u64)(x == low); },
                      [&](u64 z) { return min((u64)keep, z) - 1; });
    }
  }
  return row.walk(
      s,
      [&](float x, int i) {
        return x > low || (x == low && i <= last) ? w(x) : 0;
      },
      [&](u64 z) { return (u64)((double)uniform * (double)z); });
}

struct Options {
  float t, p, uniform, hi, lo;    // hi + lo = log2(e) / temperature
  int k;                          // 0: no cut
  DEV Weight weight(float mx) const { return {mx, hi, lo}; }
};

DEV Options options_of(long b, const float* temperature, const float* top_p,
                       const int* top_k, const float* uniform, int vocab) {
  Options o;
  o.t = temperature[b];
  o.p = top_p[b];
  o.uniform = uniform[b];
  const int k = top_k[b];
  o.k = k > 0 && k < vocab ? k : 0;
  const double c = 1.4426950408889634 / (double)fmaxf(o.t, 1e-6f);
  o.hi = (float)c;
  o.lo = (float)(c - (double)o.hi);
  return o;
}

template <typename T, bool VEC>
__global__ __launch_bounds__(NT) void sample_kernel(
    long* __restrict__ out, const T* __restrict__ logits,
    const float* __restrict__ temperature, const float* __restrict__ top_p,
    const int* __restrict__ top_k, const float* __restrict__ uniform,
    int vocab) {
  __shared__ Scratch s;
  const int tid = threadIdx.x;
  const long b = blockIdx.x;
  Row<T, VEC> row{logits + b * vocab, vocab, true};

  // the largest value, where its first 8 values are, and the smallest; neither
  // is that of a NaN
  float mx = -INFINITY, mn = INFINITY;
  int at = vocab;
  row.each8([&](const float* x, int i) {
    const float m = largest(x);
    if (m > mx && mx < FLT_MAX) {
      mx = fminf(m, FLT_MAX);
      at = i;
    }
    if constexpr (VEC) {
      const float n = smallest(x);
      if (i < vocab) mn = fminf(mn, n);
    } else {
      #pragma unroll
      for (int j = 0; j < 8; ++j)
        if (x[j] >= -FLT_MAX) mn = fminf(mn, x[j]);
    }
  });
  const float own = mx;
  best_of_all(s, mx, at, mn);
  mn = fminf(mn, mx);
  const Options o = options_of(b, temperature, top_p, top_k, uniform, vocab);
  if (o.t == 0.f || !(mx >= -FLT_MAX)) {        // or there is no value
    if (tid == 0)
      out[b] = greedy_index(row.p, mx, at, vocab,
                            o.t == 0.f ? 0 : vocab - 1);
    return;
  }
  row.finite = mx < FLT_MAX;
  const Weight w = o.weight(mx);
  if (o.p < 1.f && !(o.p > 0.f)) {              // nothing stays
    if (tid == 0) out[b] = vocab - 1;
    return;
  }
  u64 kept = 0;
  // a share is not looked for where many threads' largest values weigh more
  // than 2^-7 of the largest: the list would be too short
  const bool few = o.k
      ? o.k <= LIST / 2
      : o.p < 1.f && __syncthreads_count((own - mx) * w.hi > -7.f) <= 2 * FEW;
  if (few && draw_from_few(s, row, w, own, o.k, o.p, o.uniform, &kept, out + b))
    return;
  __syncthreads();
  const int drawn =
      draw_from_row(s, row, w, mn, o.hi, o.k, o.p, o.uniform, kept);
  if (tid == 0) out[b] = drawn;
}

// ---- rows in slices -------------------------------------------------------
// A row a workgroup leaves most of the chip idle.  Here a row is divided into
// slices of a workgroup each, which read their values once; what they find out
// meets in a second kernel, a workgroup a row, with the largest values of each.
// Weights are relative to the slice's own largest value, so that no slice waits for
// another one; the sums of 512 values are exact, and are brought to the row's largest
// value by one factor a slice.
constexpr int HELD = 4;           // 8 values each, that a thread has (wave_sums)
constexpr int SLICES = 16;        // of a row at most
constexpr int UNITS = 4;          // a thread of the second kernel has at most
constexpr int CHUNKS = HELD * 16; // 512 values of a wave each
constexpr int NEAR = 256;         // values that are listed of a row
constexpr int SHARE = 64;         // among so many a share is looked for first

struct Slice {
  u64 mass[CHUNKS];               // weights of the chunks, where asked for
  float mx, mn;                   // largest (-inf: no value), smallest
  int at;                         // first of the 8 with the first largest
  float low;                      // values from it on are listed
  int n;                          // as many
  int list_at[NEAR];
  float list[NEAR];
  float own[NT];                  // largest values of the threads, or of 2 or 4
};

// threads of a slice whose values are looked at together
DEV int together(int slices) { return slices <= 4 ? 1 : slices <= 8 ? 2 : 4; }

// Whether slices list values for top_k (0: there is none).  Up to 100: of more, the
// row's list is too long now and then (128 of 16, 64 and 240 rows 16.6 16.7 16.3 ->
// 17.5 17.8 17.9 us, 100 of 64 15.4 -> 14.6).
DEV bool listed_k(int k) { return k > 0 && k <= 100; }

constexpr int COUNTS = 256;       // steps that a slice's threads are counted in

// From s.count, how many threads' largest values are in each of COUNTS steps: the
// end of the step in which `want` of them are reached, COUNTS + 1 if there are
// fewer, how many are up to there, and how many up to about step `near`.  Each wave by
// itself, 4 steps a lane.
struct Reached {
  int end;
  unsigned n, near;
};
DEV Reached end_of(const Scratch& s, unsigned want, int near) {
  const int lane = threadIdx.x & 63;
  const uint4 c = reinterpret_cast<const uint4*>(s.count)[lane];
  const unsigned upto = wave_scan(c.x + c.y + c.z + c.w);
  const unsigned nearer = lane_of(upto, min(near / 4, 63));
  const u64 there = __ballot(upto >= want);
  if (!there) return {COUNTS + 1, lane_of(upto, 63), nearer};
  int end = lane * 4 + 4;
  unsigned n = upto;
  if (n - c.w >= want) {
    n -= c.w;
    --end;
    if (n - c.z >= want) {
      n -= c.z;
      --end;
      if (n - c.y >= want) {
        n -= c.y;
        --end;
      }
    }
  }
  const int first = __ffsll(there) - 1;
  return {lane_of(end, first), lane_of(n, first), nearer};
}

// Steps below the largest value, down to where weights are zero
struct Steps {
  float mx, zero, range, scale;
  bool whole;                     // down to there, and not only to the smallest
  DEV void between(float largest, float mn, float hi, int steps) {
    mx = largest;
    zero = 43.f / hi;
    range = mn >= -FLT_MAX ? fminf(mx - mn, zero) : zero;
    scale = (float)steps * __builtin_amdgcn_rcpf(fmaxf(range, 1e-30f));
    whole = range >= zero;
  }
  DEV float of(float x) const { return (mx - x) * scale; }
};

template <typename T, bool VEC>
__global__ __launch_bounds__(NT) void sample_slice_kernel(
    Slice* __restrict__ slice, const T* __restrict__ logits,
    const float* __restrict__ temperature, const float* __restrict__ top_p,
    const int* __restrict__ top_k, int vocab, int slices, int span) {
  __shared__ Scratch s;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const long b = blockIdx.x / slices;
  const int first = (int)(blockIdx.x % slices) * span;
  const int end = min(first + span, vocab);
  Slice& mine = slice[blockIdx.x];
  Row<T, VEC> row{logits + b * vocab, vocab, true};
  typename Row<T, VEC>::Raw raw[HELD];
  #pragma unroll
  for (int q = 0; q < HELD; ++q)
    row.hold(first + (q * NT + tid) * 8, end, raw[q]);
  const Options o = options_of(b, temperature, top_p, top_k, temperature,
                               vocab);
  s.count[tid] = 0;
  if (tid == 0) s.n = 0;
  float mx = -INFINITY, mn = INFINITY;
  int at = vocab;
  float top[HELD];                // largest of each 8
  #pragma unroll
  for (int q = 0; q < HELD; ++q) {
    const int i = first + (q * NT + tid) * 8;
    float x[8];
    row.spread(raw[q], x);
    const float m = top[q] = largest(x), n = smallest(x);
    if (m > mx && mx < FLT_MAX) {
      mx = fminf(m, FLT_MAX);
      at = i;
    }
    if (i + 8 <= end) mn = fminf(mn, n);
  }
  const float thread_mx = mx;
  float own = mx;
  const int group = together(slices);
  for (int i = 1; i < group; i <<= 1) own = fmaxf(own, __shfl_xor(own, i));
  if (tid % group == 0) mine.own[tid / group] = own;
  best_of_all(s, mx, at, mn);
  if (tid == 0) {
    mine.mx = mx;
    mine.mn = mn;
    mine.at = at;
  }
  if (o.t == 0.f || !(mx >= -FLT_MAX)) {
    if (tid < CHUNKS) mine.mass[tid] = 0;
    if (tid == 0) {
      mine.low = -INFINITY;
      mine.n = 0;
    }
    return;
  }
  // What is listed: for top_k as many values as a slice has where the k largest
  // are spread by chance, and 4 times the root of that (with 3 times a row in 16
  // slices had less than k in them now and then: 16 rows with top_k 50 12.2 -> 13.8
  // us), or all that have weight; for a share the same of SHARE, but none of less
  // than 2^-16 of the largest.
  const bool listing = o.k ? listed_k(o.k) : o.p < 1.f;
  Steps steps;
  float last = COUNTS;
  if (listing) {
    steps.between(mx, mn, o.hi, COUNTS);
    if (!o.k) last = fminf(16.f / 43.f * steps.zero * steps.scale, COUNTS);
    const float step = steps.of(thread_mx);
    if (step < last) atomicAdd(&s.count[(int)step], 1u);
  }
  row.finite = mx < FLT_MAX;
  if (!o.k) {
    const Weight w = o.weight(mx);
    u64 sum[HELD];
    #pragma unroll
    for (int q = 0; q < HELD; ++q) {
      float x[8];
      row.spread(raw[q], x);
      u64 z = 0;
      // 8 weights of less than 2^-12 are a sum of 32 bits
      if (__all(!((top[q] - mx) * w.hi >= -12.f))) {
        unsigned of8 = 0;
        if (w.any(top[q]))
          #pragma unroll
          for (int i = 0; i < 8; ++i) of8 += w.small(x[i]);
        z = of8;
      } else if (w.any(top[q])) {
        #pragma unroll
        for (int i = 0; i < 8; ++i) z += w.always(x[i]);
      }
      sum[q] = z;
    }
    const u64 z = wave_sums(sum);
    if (lane < HELD) mine.mass[lane * 16 + wid] = z;
  }
  const float none = from_ordered(ordered(mx) + 1);
  if (!listing) {
    if (tid == 0) {
      mine.low = none;
      mine.n = 0;
    }
    return;
  }
  __syncthreads();
  const float part = (float)(o.k ? o.k : SHARE) *
                     __builtin_amdgcn_rcpf((float)slices);
  const Reached reached =
      end_of(s, (unsigned)(part + 4.f * __builtin_amdgcn_sqrtf(part)) + 2,
             (int)fminf(7.f / 43.f * steps.zero * steps.scale, COUNTS));
  const float low = reached.end > COUNTS && o.k && !steps.whole
      ? none
      : fmaxf(mx - fminf((float)reached.end, last) * (steps.range / COUNTS),
              -FLT_MAX);
  // Too many values, or a share where the largest of more than 2 FEW threads weigh more
  // than 2^-7 of the slice's, as below: without a look at each of them.  us before
  // lists, with lists and so: share of normal logits 64 rows of 128256 118 120 118, 240
  // of 32768 48.5 50.6 48.6, top_k 50 of logits of 4 values 155 161 157, 52 58 54
  const int most = NEAR / group;
  if ((int)reached.n > most || !o.k && reached.near > 2 * FEW) {
    if (tid == 0) {
      mine.low = none;
      mine.n = 0;
    }
    return;
  }
  // a thread has few, so each goes through its own: one of its 8 values, and
  // one of these
  unsigned loads = 0;
  #pragma unroll
  for (int q = 0; q < HELD; ++q) loads |= (top[q] >= low) << q;
  for (; loads; loads &= loads - 1) {
    const int q = __ffs(loads) - 1;
    auto r = raw[0];
    #pragma unroll
    for (int j = 1; j < HELD; ++j)
      if (q == j) r = raw[j];
    float x[8];
    row.spread(r, x);
    unsigned hits = 0;
    #pragma unroll
    for (int i = 0; i < 8; ++i) hits |= (x[i] >= low) << i;
    for (; hits; hits &= hits - 1) {
      const int i = __ffs(hits) - 1;
      float y = x[0];
      #pragma unroll
      for (int j = 1; j < 8; ++j) y = i == j ? x[j] : y;
      const int n = (int)atomicAdd(&s.n, 1u);
      if (n >= most) {
        loads = 0;
        break;
      }
      mine.list[n] = y;
      mine.list_at[n] = first + (q * NT + tid) * 8 + i;
    }
  }
  __syncthreads();
  if (tid == 0) {
    mine.low = (int)s.n <= most ? low : none;
    mine.n = (int)s.n <= most ? (int)s.n : 0;
  }
}

template <typename T, bool VEC>
__global__ __launch_bounds__(NT) void sample_slices_kernel(
    long* __restrict__ out, const Slice* __restrict__ slice,
    const T* __restrict__ logits, const float* __restrict__ temperature,
    const float* __restrict__ top_p, const int* __restrict__ top_k,
    const float* __restrict__ uniform, int vocab, int slices, int span) {
  __shared__ Scratch s;
  __shared__ int unit[LIST];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const long b = blockIdx.x;
  slice += b * slices;
  Row<T, VEC> row{logits + b * vocab, vocab, true};
  // All loads are issued before anything waits: chunk `tid` of the row, a value
  // that a slice lists, the largest values of UNITS units, and by lane i of 16 what
  // slice i says.
  const u64 chunk = slice[min(tid / CHUNKS, slices - 1)].mass[tid % CHUNKS];
  const int group = together(slices), most = NEAR / group;
  // all of a wave are in one list
  const int from_list = __builtin_amdgcn_readfirstlane(tid / most);
  const Slice& listing = slice[min(from_list, slices - 1)];
  const float x = listing.list[tid % most];
  const int x_at = listing.list_at[tid % most];
  const int each = NT / group;  // units a slice
  float own[UNITS];
  #pragma unroll
  for (int q = 0; q < UNITS; ++q) {
    const int i = q * NT + tid;
    own[q] = i < slices * each ? slice[i / each].own[i % each] : -INFINITY;
  }
  const Slice& head = slice[min(lane & 15, slices - 1)];
  const float slice_mx = head.mx;
  const int slice_n = head.n;
  float mx = slice_mx, mn = head.mn, low = head.low;
  int at = head.at;
  const Options o = options_of(b, temperature, top_p, top_k, uniform, vocab);
  const u64 best = lane_of(
      row_scan((u64)ordered(mx + 0.f) << 32 | (unsigned)~at, u64(0),
               [](u64 a, u64 b) { return a > b ? a : b; }), 15);
  mx = from_ordered((unsigned)(best >> 32));
  at = (int)~(unsigned)best;
  if (o.t == 0.f || !(mx >= -FLT_MAX)) {
    if (tid == 0)
      out[b] = greedy_index(row.p, mx, at, vocab, o.t == 0.f ? 0 : vocab - 1);
    return;
  }
  if (o.p < 1.f && !(o.p > 0.f)) {              // nothing stays
    if (tid == 0) out[b] = vocab - 1;
    return;
  }
  const Weight w = o.weight(mx);
  u64 mass = 0, upto = 0;         // of the wave's chunks, which are of one slice
  if (!o.k && wid < slices) {
    const double factor = exp2(((double)lane_of(slice_mx, wid) - (double)mx) *
                               ((double)o.hi + (double)o.lo));
    if (chunk) mass = (u64)rint((double)chunk * factor);
    upto = wave_scan(mass);
  }
  if (lane == 63) s.wave_mass[wid] = upto;
  if (!o.k && !(o.p < 1.f)) {
    __syncthreads();
    u64 z;
    const u64 before = sum_of_16(s.wave_mass, wid, &z);
    // the token is in the chunk where the running sum passes the target;
    // there sums are those of the slice's own weights again
    const u64 target = (u64)((double)o.uniform * (double)z);
    if (target >= z) {
      if (tid == 0) out[b] = vocab - 1;
      return;
    }
    // a wave has the chunks of one slice, in the order of its values
    const u64 over = __ballot(before + upto > target);
    if (before > target || !over) return;
    const int i = __ffsll(over) - 1, of = wid;
    const u64 all = __shfl(chunk, i);
    const double part = (double)(target - before - __shfl(upto - mass, i)) /
                        (double)__shfl(mass, i);
    const u64 goal = min((u64)(part * (double)all), all - 1);
    const Weight wi = o.weight(__shfl(slice_mx, of));
    row.finite = wi.mx < FLT_MAX;
    const int stop = min((of + 1) * span, vocab);
    const int from = of * span + i * 512 + lane * 8;
    typename Row<T, VEC>::Raw raw;
    row.hold(from, stop, raw);
    float x[8];
    row.spread(raw, x);
    u64 sum = 0;
    #pragma unroll
    for (int j = 0; j < 8; ++j) sum += wi.always(x[j]);
    const u64 mine = wave_scan(sum);
    const u64 here = __ballot(mine > goal);
    if (lane == __ffsll(here) - 1) {
      u64 c = mine - sum;
      int found = 0;
      #pragma unroll
      for (int j = 0; j < 8; ++j) {
        c += wi.always(x[j]);
        found += c <= goal;
      }
      out[b] = from + found;
    }
    return;
  }
  // What the slices list of the values from the highest of their ends on is all
  // that the row has of them.
  low = lane_of(row_scan(low, -INFINITY, [](float a, float b) {
    return fmaxf(a, b);
  }), 15);
  const bool listed = from_list < slices && x >= low &&
                      tid % most < lane_of(slice_n, from_list & 15);
  const u64 lanes = __ballot(listed);
  u64 x_mass = 0, list_mass = 0;
  if (lanes) {
    x_mass = listed ? w(x) : 0;
    if (!o.k) list_mass = wave_scan(x_mass);
  }
  if (lane == 63) {
    s.list_mass[wid] = list_mass;
    s.wave_count[wid] = __popcll(lanes);
  }
  if (tid == 0) s.n = s.keep = s.stay = 0;
  s.count[tid] = 0;
  __syncthreads();
  u64 z = 0, part = 0;            // weight of all
  unsigned n;
  const int place = (int)sum_of_16(s.wave_count, wid, &n) +
                    __popcll(lanes & ((u64(1) << lane) - 1));
  bool done = n > 0 && n <= NEAR;
  if (o.k) {
    // or below the list there is no weight
    done = done && ((int)n >= o.k || !w.any(low));
  } else {
    z = sum_of_16(s.wave_mass);
    part = part_of(o.p, z);
    done = done && sum_of_16(s.list_mass) >= part;
  }
  if (done) {
    if (listed) s.entry[place] = {key_of(x, x_at), x_mass};
    __syncthreads();
    draw_from_entries(s, (int)n, vocab, o.k, o.p, o.uniform, part, out + b);
    return;
  }
  // The draw where all that stays is among few values: the want-th largest of
  // the units' largest values has at least that many values at or above it, and
  // hardly more.  A share is not looked for where many units' largest values
  // weigh more than 2^-7 of the largest: the list would be too short.
  mn = fminf(lane_of(row_scan(mn, INFINITY, min_of), 15), mx);
  row.finite = mx < FLT_MAX;
  int near = 0;
  #pragma unroll
  for (int q = 0; q < UNITS; ++q)
    near += __popcll(__ballot((own[q] - mx) * w.hi > -7.f));
  Steps steps;
  steps.between(mx, mn, w.hi, NT);
  if (lane == 0) atomicAdd(&s.n, (unsigned)near);
  #pragma unroll
  for (int q = 0; q < UNITS; ++q) {
    const float step = steps.of(own[q]);
    if (step < (float)NT) atomicAdd(&s.count[(int)step], 1u);
  }
  __syncthreads();
  if (o.k ? o.k <= LIST / 2 : s.n <= 2 * FEW) {
    const unsigned want = o.k ? o.k : FEW, upto = wave_scan(s.count[tid]);
    if (lane == 63) s.wave_count[wid] = upto;
    if (tid == 0) s.step = NT + 1;
    __syncthreads();
    unsigned all;
    const unsigned before = sum_of_16(s.wave_count, wid, &all);
    if (before + upto >= want && before + upto - s.count[tid] < want)
      s.step = tid + 1;
    __syncthreads();
    // NT + 1: fewer units than wanted are in the steps.  Then every value that
    // has weight may stay, the smallest ones, which no step has, among them.
    const float end = s.step <= NT || steps.whole ? (float)s.step : INFINITY;
    #pragma unroll
    for (int q = 0; q < UNITS; ++q)
      if (steps.of(own[q]) < end) {
        const unsigned n = atomicAdd(&s.keep, 1u);
        if (n < LIST) unit[n] = q * NT + tid;
      }
    __syncthreads();
    const int units = (int)s.keep;
    if (tid == 0) s.n = 0;
    __syncthreads();
    if (units <= LIST) {
      // loads of 8 values: of `group` threads, as often as those loaded
      const int loads = group * ((span + NT * 8 - 1) / (NT * 8));
      for (int i = tid; i < units * loads; i += NT) {
        const int u = unit[i / loads], j = i % loads, of = u / each;
        const int from = of * span +
            (j / group * NT + u % each * group + j % group) * 8;
        typename Row<T, VEC>::Raw raw;
        row.hold(from, min((of + 1) * span, vocab), raw);
        float x[8];
        row.spread(raw, x);
        #pragma unroll
        for (int v = 0; v < 8; ++v)
          if (steps.of(x[v]) < end) {
            const unsigned n = atomicAdd(&s.n, 1u);
            if (n < LIST) {
              s.list[n] = x[v];
              s.list_at[n] = from + v;
            }
          }
      }
      __syncthreads();
      if (draw_from_list(s, w, vocab, o.k, o.p, o.uniform, z, out + b)) return;
    }
  }
  __syncthreads();
  const int drawn =
      draw_from_row(s, row, w, mn, o.hi, o.k, o.p, o.uniform, z);
  if (tid == 0) out[b] = drawn;
}

// Slices of a row, 0: none (or no rows).  As many as give every compute unit a
// workgroup, if each has a load for every thread.  Beyond two workgroups a unit the
// chip is full of whole rows.  A mix of options would gain in slices there (us, 256
// rows of 128256 43, in 4 slices 39, 384 of 50257 in 2 83 59), but rows that are all
// greedy (13 and 20) and shares of thousands of values (132 and 147) lose, and weights
// relative to a slice's largest value are other last bits, which decide a draw now
// and then.
int sample_slices(long rows, int vocab) {
  const int least = (vocab + HELD * NT * 8 - 1) / (HELD * NT * 8);
  const int most = min(SLICES, max(1, vocab / (NT * 8)));
  if (rows == 0 || least > SLICES || rows * least > 512) return 0;
  return max(least, min(most, (int)(256 / rows)));
}

}  // namespace

// bytes of the workspace, 0: none is needed
long sample_workspace(long rows, int vocab) {
  return rows * sample_slices(rows, vocab) * (long)sizeof(Slice);
}

// ws null: a workgroup a row
template <typename T>
void launch_sample(long* out, const T* logits, const float* temperature,
                   const float* top_p, const int* top_k, const float* uniform,
                   void* ws, long rows, int vocab, hipStream_t stream) {
  if (rows == 0) return;
  const bool vec = vocab % 8 == 0 && reinterpret_cast<size_t>(logits) % 16 == 0;
  const int slices = ws ? sample_slices(rows, vocab) : 0;
  const int span = slices ? ((vocab + slices - 1) / slices + 7) / 8 * 8 : 0;
  Slice* slice = static_cast<Slice*>(ws);
  #define RUN(VEC)                                                          \
    if (slices) {                                                           \
      sample_slice_kernel<T, VEC>                                           \
          <<<(unsigned)(rows * slices), NT, 0, stream>>>(                   \
              slice, logits, temperature, top_p, top_k, vocab, slices,      \
              span);                                                        \
      sample_slices_kernel<T, VEC><<<(unsigned)rows, NT, 0, stream>>>(      \
          out, slice, logits, temperature, top_p, top_k, uniform, vocab,    \
          slices, span);                                                    \
    } else {                                                                \
      sample_kernel<T, VEC><<<(unsigned)rows, NT, 0, stream>>>(             \
          out, logits, temperature, top_p, top_k, uniform, vocab);          \
    }
  if (vec) {
    RUN(true)
  } else {
    RUN(false)
  }
  #undef RUN
}
template void launch_sample<bf16>(long*, const bf16*, const float*,
                                  const float*, const int*, const float*,
                                  void*, long, int, hipStream_t);
template void launch_sample<float>(long*, const float*, const float*,
                                   const float*, const int*, const float*,
                                   void*, long, int, hipStream_t);

template <typename T>
void launch_greedy_sample(long* out, const T* logits, long rows, int vocab,
                          hipStream_t stream) {
  greedy_sample_kernel<T><<<dim3((unsigned)rows), 256, 0, stream>>>(
      out, logits, vocab);
}
template void launch_greedy_sample<bf16>(long*, const bf16*, long, int,
                                         hipStream_t);
template void launch_greedy_sample<float>(long*, const float*, long, int,
                                          hipStream_t);
