// Integer arithmetic of the classic launch, for the kernels, for the host code
// that prepares their arguments and (tests/test_launch_division.py) for a plain
// C++ compiler: division by an invariant, and the token ranges of a sequence's
// splits.
#ifndef PA_LAUNCH_MATH_H_
#define PA_LAUNCH_MATH_H_

#include <stdint.h>

#include <algorithm>

#ifdef __HIP__
#define PA_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define PA_HOST_DEVICE inline
#endif

constexpr int kSplitAlign = 32;    // split ranges are multiples of this many tokens

// Division of an n < 2^31 by a d that the host knows: floor(n / d) = n * mul >>
// (32 + shift), mul = floor(2^(31 + l) / d) + 1, l = ceil(log2 d), shift = l -
// 1 (Granlund and Montgomery's division by an invariant). A general 32-bit
// division is ~25 dependent instructions in front of a kernel's first loads
// and a 64-bit one ~150; with these the classic split's two kernels start
// their loads 0.4 us earlier: whole calls at the Llama-3-8B shape, graph-timed,
// B = 1, T = 2048 8.7 -> 8.3 us, B = 8, T <= 2500 17.0 -> 16.5, unsplit B = 24,
// T <= 192 (Qwen2.5-0.5B shape) 4.66 -> 4.49.
struct Div {
  uint32_t d, mul, shift;
};

inline Div make_div(uint32_t d) {
  Div v = {d, 0, 0};
  if (d > 1) {
    const uint32_t l = 32 - __builtin_clz(d - 1);
    v.mul = (uint32_t)((uint64_t(1) << (31 + l)) / d + 1);
    v.shift = l - 1;
  }
  return v;
}

PA_HOST_DEVICE uint32_t div_by(uint32_t n, const Div &v) {
  return v.d == 1 ? n : (uint32_t)((uint64_t)n * v.mul >> 32) >> v.shift;
}

// The classic split's division of a sequence: tiles of a split of max_seq_len
// tokens (0: not given), and the divisors.
struct SplitDiv {
  int32_t max_seq_len, chunk_tiles;
  Div by_splits, by_chunk;
};

inline SplitDiv split_div(int max_seq_len, int num_splits) {
  const uint32_t tiles = ((uint32_t)max_seq_len + kSplitAlign - 1) / kSplitAlign;
  SplitDiv s;
  s.max_seq_len = max_seq_len;
  s.chunk_tiles = (int)((tiles + num_splits - 1) / num_splits);
  s.by_splits = make_div(num_splits);
  s.by_chunk = make_div(std::max(1, s.chunk_tiles));
  return s;
}

// Token range [lo, hi) of one split, and how many of the sequence's splits
// hold tokens. chunk = ceil(ceil(T / 32) / S) * 32 tokens, T = the sequence's
// length (the reference's per-sequence rule, triton_decode.py:78-85), or the
// chunk of a max_seq_len-token sequence when max_seq_len > 0 and that is
// larger (ragged batches: long sequences take all S splits, short ones few;
// never below the sequence's own chunk, so no token is dropped).
struct SplitRange {
  int lo, hi, n;
};

PA_HOST_DEVICE SplitRange split_range(int seq_len, const SplitDiv &p, int split) {
  static_assert(kSplitAlign == 32, "lengths are counted in 32-token tiles");
  auto least = [](uint32_t a, uint32_t b) { return a < b ? a : b; };
  auto most = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
  const uint32_t tiles = ((uint32_t)seq_len + 31) >> 5;  // < 2^27
  uint32_t chunk = (uint32_t)p.chunk_tiles;
  uint32_t n;
  if (chunk != 0 && seq_len <= p.max_seq_len) {
    n = div_by(tiles + chunk - 1, p.by_chunk);
  } else {
    // T = 0 still has one split
    chunk = most(most(div_by(tiles + p.by_splits.d - 1, p.by_splits), chunk), 1u);
    n = (tiles + chunk - 1) / chunk;
  }
  const uint32_t lo = least((uint32_t)split * chunk, tiles);
  SplitRange r;
  r.lo = (int)least(lo << 5, (uint32_t)seq_len);
  r.hi = (int)least(least(lo + chunk, tiles) << 5, (uint32_t)seq_len);
  r.n = (int)n > 1 ? (int)n : 1;
  return r;
}

#endif  // PA_LAUNCH_MATH_H_
