// Sampling kernels: greedy argmax, and the whole of temperature, top-k, top-p
// and draw.
//
// One workgroup per batch row over vocab-size logits (128256 for Llama-3).
// Vectorized bf16/f32 reads; fp32 math, sums of weights in 64-bit integers.
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
// What bounds it: vector instructions on every value, in passes over the row,
// which stays in L2: 8 us for the largest, 20 for the weights of 128256.  So 8
// values are looked at together where that decides about all of them.  Where
// few values stay, and next-token logits have a few dozen that matter, they are
// listed in the second pass and the rest is done on the list, up to 8 threads a
// value.  Otherwise no sort either: one histogram of counts and weights over
// 2048 equal steps between the largest and the smallest logit finds the step
// where the wanted count or share is reached, and ranks the few values in it
// exactly (or divides that step again).  Equal steps of the logit, and not
// digits of its bit pattern, because next-token logits fill few exponents: 64
// lanes that add to the same few counters in LDS would go one by one.
//
// 64 rows of 128256, 48 values far above the others, us with the histogram
// alone and now: greedy 15 11, temperature 57 38, top_p 0.9 115 39, top_k 50
// 85 27, top_k 40 and top_p 141 28; a mix 138 45, where the library's sorts,
// scans and selections took 2625.  Normal logits, whose share is thousands of
// values, 155 132.
//
// Weights are 2^-40 fixed point relative to the largest, so every sum is
// exact, does not depend on its order, and the same inputs give the same
// token.
namespace {

typedef unsigned long long u64;
constexpr int NT = 1024;          // threads
constexpr int STEPS = 2048;       // of the histogram
constexpr int LIST = 512;         // values ranked one by one
constexpr int AHEAD = 2;          // loads of a thread on their way
constexpr int FEW = 128;          // values that a share is looked for in

struct Weight {
  float mx, hi, lo;               // hi + lo = log2(e) / temperature
  // false: weights of x and less are below half of 2^-40
  DEV bool any(float x) const { return (x - mx) * hi > -42.f; }
  DEV u64 operator()(float x) const {
    if (!any(x)) return 0;
    const float d = x - mx, t = d * hi;
    const float r = fmaf(d, hi, -t) + d * lo;
    float e = __builtin_amdgcn_exp2f(t);
    e = fmaf(e * r, 0.69314718f, e) * 1099511627776.f + 0.5f;
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

template <typename I> DEV I wave_scan(I x) {      // inclusive
  const int lane = threadIdx.x & 63;
  #pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const I v = __shfl_up(x, o);
    if (lane >= o) x += v;
  }
  return x;
}

struct Scratch {
  u64 mass[STEPS];
  unsigned count[STEPS];
  float list[LIST];
  u64 list_mass[LIST];
  int list_at[LIST];
  u64 wave_mass[16];
  unsigned wave_count[16];
  u64 before_mass, kept_mass;
  unsigned before_count, n, key_min, key_max, keep;
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

  // First index at which the running sum of w(x, index) exceeds the target
  // that `of` makes of the whole sum; vocab - 1 if there is none.  A wave has a
  // sixteenth; the one where the target lies is divided again.
  template <typename W, typename F>
  DEV int walk(Scratch& s, W w, F of) const {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int first = 0, end = vocab;
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
          s.list_mass[at] = w(x);
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
        const u64 one = s.list_mass[tid];
        u64 mb = mass0;
        unsigned cb = count0, equal = 0;
        for (unsigned j = 0; j < members; ++j) {
          const float y = s.list[j];
          equal += y == x;
          if (y > x) {
            mb += s.list_mass[j];
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

// The draw where all that stays is among few values: the want-th largest of the
// threads' own largest values has at least that many values at or above it, and
// hardly more.  Those are listed in one pass, ranked, and the token is drawn
// from the list.  k 0: no top_k, and `all` is the weight of all values.  False
// if the list is too short for the share or too long.
template <typename R>
DEV bool draw_from_few(Scratch& s, const R& row, const Weight& w, float own,
                       int k, float p, float u, u64* all, int* drawn) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int want_n = k > 0 ? k : FEW;
  const unsigned key = ordered(own);
  unsigned prefix = 0;            // 16 bits are close enough
  for (int bit = 31; bit >= 16; --bit) {
    const unsigned next = prefix | 1u << bit;
    if (__syncthreads_count(key >= next) >= want_n) prefix = next;
  }
  const float least =
      prefix > ordered(-FLT_MAX) ? from_ordered(prefix) : -FLT_MAX;
  if (tid == 0) {
    s.n = 0;
    s.value = -INFINITY;
  }
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
  z = wave_scan(z);
  if (lane == 63) s.wave_mass[wid] = z;
  __syncthreads();
  const int n = (int)s.n;
  z = 0;
  for (int v = 0; v < 16; ++v) z += s.wave_mass[v];
  *all = z;
  if (tid < n && n <= LIST) s.list_mass[tid] = w(s.list[tid]);
  __syncthreads();
  if (n > LIST) return false;
  // `share` neighbouring threads a value, each with a part of the others
  const int share = n <= NT / 8 ? 8 : n <= NT / 4 ? 4 : 2;
  const int mine = tid / share, part = tid % share;
  const bool one_of = mine < n;
  auto sum = [&](auto v) {
    for (int o = 1; o < share; o <<= 1) v += __shfl_xor(v, o);
    return v;
  };
  float x = -INFINITY;
  int index = 0;
  u64 one = 0, above = 0;
  int before = 0, equal = 0, earlier = 0;
  if (one_of) {
    x = s.list[mine];
    index = s.list_at[mine];
    one = s.list_mass[mine];
    #pragma unroll 2
    for (int j = part; j < n; j += share) {
      const float y = s.list[j];
      above += y > x ? s.list_mass[j] : 0;
      before += y > x;
      equal += y == x;
      earlier += y == x && s.list_at[j] < index;
    }
  }
  above = sum(above);
  before = sum(before);
  equal = sum(equal);
  earlier = sum(earlier);
  float low = -INFINITY;
  if (k > 0) {
    if (one_of && before < k && before + equal >= k) {
      s.value = x;                // every member of the group writes the same
      s.kept_mass = above + one * equal;
    }
    __syncthreads();
    low = s.value;
    if (low > -INFINITY)
      z = s.kept_mass;
    else                          // fewer than k values: all are in the list
      for (int j = 0; j < n; ++j) z += s.list_mass[j];
  }
  int last = row.vocab;
  if (p < 1.f) {
    const u64 want = (u64)ceil((double)p * (double)z);
    if (tid == 0) s.found = -1;
    __syncthreads();
    if (one_of && x >= low && above < want && above + one * equal >= want &&
        (u64)earlier + 1 == (want - above + one - 1) / one) {
      s.value = x;
      s.found = index;
    }
    __syncthreads();
    low = s.value;
    last = s.found;
    __syncthreads();
    if (last < 0) return false;
  }
  const bool stays = one_of && (x > low || (x == low && index <= last));
  if (one_of && !stays) s.list_mass[mine] = 0;
  if (tid == 0) s.found = row.vocab - 1;
  __syncthreads();
  u64 all_kept = 0, upto = 0;
  if (stays)
    #pragma unroll 2
    for (int j = part; j < n; j += share) {
      const u64 m = s.list_mass[j];
      all_kept += m;
      upto += s.list_at[j] < index ? m : 0;
    }
  all_kept = sum(all_kept);
  upto = sum(upto);
  const u64 target = (u64)((double)u * (double)all_kept);
  if (stays && upto <= target && upto + one > target) s.found = index;
  __syncthreads();
  *drawn = s.found;
  return true;
}

template <typename T, bool VEC>
__global__ __launch_bounds__(NT) void sample_kernel(
    long* __restrict__ out, const T* __restrict__ logits,
    const float* __restrict__ temperature, const float* __restrict__ top_p,
    const int* __restrict__ top_k, const float* __restrict__ uniform,
    int vocab) {
  __shared__ Scratch s;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
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
  #pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float x = __shfl_xor(mx, o);
    const int i = __shfl_xor(at, o);
    if (x > mx || (x == mx && i < at)) {
      mx = x;
      at = i;
    }
    mn = fminf(mn, __shfl_xor(mn, o));
  }
  if (lane == 0) {
    s.list[wid] = mx;
    s.list[16 + wid] = mn;
    s.count[wid] = at;
  }
  __syncthreads();
  for (int v = 0; v < 16; ++v) {
    const float x = s.list[v];
    const int i = s.count[v];
    if (x > mx || (x == mx && i < at)) {
      mx = x;
      at = i;
    }
    mn = fminf(mn, s.list[16 + v]);
  }
  mn = fminf(mn, mx);
  __syncthreads();
  const float t = temperature[b];
  if (t == 0.f || !(mx >= -FLT_MAX)) {          // or there is no value
    if (tid == 0) {
      int first = t == 0.f ? 0 : vocab - 1;
      if (mx >= -FLT_MAX) {
        for (first = at; in_range(Elem<T>::ld(row.p + first)) != mx;)
          ++first;
      }
      out[b] = first;
    }
    return;
  }
  row.finite = mx < FLT_MAX;

  const double c = 1.4426950408889634 / (double)fmaxf(t, 1e-6f);
  const Weight w{mx, (float)c, (float)(c - (double)(float)c)};
  // below this weights are zero
  const float floor = mx - 64.f / (float)c;
  const float lo = mn >= -FLT_MAX ? fmaxf(mn, floor) : floor;
  float low = -INFINITY;          // values above it stay
  int last = -1;                  // and its equals up to this index
  u64 kept = 0;                   // their weight, 0: not known
  const int k = top_k[b];
  const float p = top_p[b];
  if (p < 1.f && !(p > 0.f)) {    // nothing stays
    if (tid == 0) out[b] = vocab - 1;
    return;
  }
  const bool cut = k > 0 && k < vocab;
  // a share is not looked for where many threads' largest values weigh more
  // than 2^-7 of the largest: the list would be too short
  if (cut ? k <= LIST / 2
          : p < 1.f && __syncthreads_count((own - mx) * w.hi > -7.f) <=
                           2 * FEW) {
    int drawn;
    if (draw_from_few(s, row, w, own, cut ? k : 0, p, uniform[b], &kept,
                      &drawn)) {
      if (tid == 0) out[b] = drawn;
      return;
    }
    __syncthreads();
  }
  if (cut) {
    reach<true>(s, row, w, lo, mx, k);
    low = s.value;
    kept = s.keep == ~0u ? 0 : s.kept_mass;
    last = vocab;
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
  const int drawn = row.walk(
      s,
      [&](float x, int i) {
        return x > low || (x == low && i <= last) ? w(x) : 0;
      },
      [&](u64 z) { return (u64)((double)uniform[b] * (double)z); });
  if (tid == 0) out[b] = drawn;
}

}  // namespace

template <typename T>
void launch_sample(long* out, const T* logits, const float* temperature,
                   const float* top_p, const int* top_k, const float* uniform,
                   long rows, int vocab, hipStream_t stream) {
  if (rows == 0) return;
  #define RUN(VEC)                                                          \
    sample_kernel<T, VEC><<<dim3((unsigned)rows), NT, 0, stream>>>(         \
        out, logits, temperature, top_p, top_k, uniform, vocab)
  if (vocab % 8 == 0 && reinterpret_cast<size_t>(logits) % 16 == 0)
    RUN(true);
  else
    RUN(false);
  #undef RUN
}
template void launch_sample<bf16>(long*, const bf16*, const float*,
                                  const float*, const int*, const float*,
                                  long, int, hipStream_t);
template void launch_sample<float>(long*, const float*, const float*,
                                   const float*, const int*, const float*,
                                   long, int, hipStream_t);

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
