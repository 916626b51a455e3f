// Host side of the BF16 context codec: encoder, decoder and rANS checkpoint
// (frame-index) builder.  Exports the C ABI the reference binds with ctypes:
//
//   bcx_encode bcx_frequencies bcx_decode bcx_decode_compact bcx_free
//   bcx_pack6 bcx_unpack6                  (GCR/bitexact_context_ans.cpp:235-359)
//   bcx_checkpoint                         (GCR/bitexact_context_gpu_index.cpp:21-26)
//   p_encode p_decode p_free               (GCR/bitexact_predictive_ans.cpp:10-12)
//   ppcx_checkpoint ppcx_checkpoint_binary (GCR/bitexact_predictive_gpu_index.cpp:9-12, 38-41)
//
// with the same argument meaning, ownership and status codes.  The
// implementation is organised differently from the reference: one table
// object (`SymbolTables`) validates the frequency rows once and answers
// slot -> symbol queries with one bucket entry (a search in the prefix sums where
// a bucket holds several symbols), and one templated walker serves
// plain decoding and checkpoint recording for both wire formats.  No function
// keeps state between calls, so all of them may run concurrently.
#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <memory>
#include <new>
#include <system_error>
#include <thread>
#include <type_traits>
#include <vector>

#include "piece_units.h"

namespace {

constexpr uint32_t kScaleBits = 16;
constexpr uint32_t kTotal = 1u << kScaleBits;
constexpr uint32_t kLow = 1u << 23;

inline uint32_t main_symbol(uint16_t w) { return (w >> 5) & 0x3FFu; }
inline uint32_t residual_symbol(uint16_t w) { return ((uint32_t)(w >> 15) << 5) | (w & 31u); }

enum class Walk { ok, abandoned, bad_context, dead_context, bad_symbol, overflow, overrun, bad_tail, bad_head };

// Validated frequency rows plus the lookup structures derived from them.
//
// A context's 65536 slots are cut into kBuckets buckets, and a bucket's entry holds the symbol that
// owns most of its slots, with the symbol's start and frequency: one load answers a query, unless a
// symbol boundary inside the bucket put the slot elsewhere (a search in the prefix sums then).
// 512 buckets: the four contexts that are live in a row of a frame (its row class by every column
// class) take 16 KiB and stay in the first-level cache with the stream, where 1024 buckets do not;
// about one query in twenty searches (a predicted branch otherwise).
class SymbolTables {
 public:
  enum class Check { ok, overflow, bad_sum };
  struct Entry {
    uint16_t symbol, start;
    uint32_t freq;  // 0 in contexts that are not live: no slot is ever inside
  };
  // A row is usable ("live") when it sums to the total.  Rows that overflow the
  // total are always an error; rows with any other sum are an error unless
  // `partial_rows_are_dead` (then they only fail when a symbol selects them).
  Check build(const uint32_t *freq, uint32_t nctx, uint32_t vocab, bool partial_rows_are_dead = false) {
    nctx_ = nctx;
    vocab_ = vocab;
    prefix_.assign((size_t)nctx * (vocab + 1), 0);
    live_.assign(nctx, 0);
    for (uint32_t c = 0; c < nctx; ++c) {
      uint32_t *p = prefix_.data() + (size_t)c * (vocab + 1);
      const uint32_t *f = freq + (size_t)c * vocab;
      uint64_t run = 0;
      for (uint32_t s = 0; s < vocab; ++s) {
        if (f[s] > kTotal || run + f[s] > kTotal) return Check::overflow;
        run += f[s];
        p[s + 1] = (uint32_t)run;
      }
      if (run != 0 && run != kTotal && !partial_rows_are_dead) return Check::bad_sum;
      live_[c] = run == kTotal;
    }
    entries_.assign((size_t)nctx * kBuckets, Entry{0, 0, 0});
    for (uint32_t c = 0; c < nctx; ++c) {
      if (!live_[c]) continue;
      const uint32_t *p = prefix_.data() + (size_t)c * (vocab + 1);
      Entry *q = entries_.data() + (size_t)c * kBuckets;
      uint32_t s = 0;
      for (uint32_t b = 0; b < kBuckets; ++b) {
        const uint32_t lo = b << kBucketShift, hi = lo + (1u << kBucketShift);
        while (p[s + 1] <= lo) ++s;
        uint32_t best = s, most = 0;
        for (uint32_t k = s; p[k] < hi; ++k) {
          const uint32_t held = std::min(p[k + 1], hi) - std::max(p[k], lo);
          if (held > most) best = k, most = held;
          if (p[k + 1] >= hi) break;
        }
        q[b] = Entry{(uint16_t)best, (uint16_t)p[best], p[best + 1] - p[best]};
      }
    }
    return Check::ok;
  }
  bool live(uint32_t c) const { return live_[c] != 0; }
  uint32_t nctx() const { return nctx_; }
  const Entry *entries() const { return entries_.data(); }
  // symbol whose half-open slot range contains `slot`, by a scan from symbol `s`; context must be live
  Entry find(uint32_t c, uint32_t slot, uint32_t s) const {
    const uint32_t *p = prefix_.data() + (size_t)c * (vocab_ + 1);
    while (p[s] > slot) --s;
    while (p[s + 1] <= slot) ++s;
    return Entry{(uint16_t)s, (uint16_t)p[s], p[s + 1] - p[s]};
  }
  const Entry &bucket(uint32_t c, uint32_t slot) const {
    return entries_[((size_t)c << kBucketBits) + (slot >> kBucketShift)];
  }
  static constexpr uint32_t kBucketBits = 9, kBuckets = 1u << kBucketBits, kBucketShift = kScaleBits - kBucketBits;

 private:
  uint32_t nctx_ = 0, vocab_ = 0;
  std::vector<uint32_t> prefix_;
  std::vector<Entry> entries_;
  std::vector<uint8_t> live_;
};

inline bool read_head(const uint8_t *s, size_t bytes, uint32_t &state) {
  if (bytes < 4) return false;
  state = (uint32_t)s[0] | (uint32_t)s[1] << 8 | (uint32_t)s[2] << 16 | (uint32_t)s[3] << 24;
  return state >= kLow;
}

struct Position {
  uint32_t state;
  size_t ip;
};

// `count` symbols from `at`, every one checked: contexts, stream bounds, state overflow.
template <class ContextFn>
Walk walk_checked(const SymbolTables &t, const uint8_t *stream, size_t bytes, ContextFn context, uint32_t count,
                  Position &at, uint16_t *out) {
  for (uint32_t i = 0; i < count; ++i) {
    const uint32_t c = context(i);
    if (c >= t.nctx()) return Walk::bad_context;
    if (!t.live(c)) return Walk::dead_context;
    const uint32_t slot = at.state & (kTotal - 1);
    const SymbolTables::Entry e = t.find(c, slot, t.bucket(c, slot).symbol);
    out[i] = e.symbol;
    const uint64_t next = (uint64_t)e.freq * (at.state >> kScaleBits) + (slot - e.start);
    if (next > std::numeric_limits<uint32_t>::max()) return Walk::overflow;
    at.state = (uint32_t)next;
    while (at.state < kLow) {
      if (at.ip >= bytes) return Walk::overrun;
      at.state = (at.state << 8) | stream[at.ip++];
    }
  }
  return Walk::ok;
}

// value < limit ? then : otherwise, as a conditional move (left alone the compiler branches, which
// mispredicts on half of the symbols).
template <uint32_t limit>
inline uint32_t select_below(bool below, uint32_t value, uint32_t then, uint32_t otherwise) {
#if defined(__x86_64__)
  (void)below;
  asm("cmpl %[limit], %[value]\n\tcmovb %[then], %[result]"
      : [result] "+r"(otherwise)
      : [value] "r"(value), [limit] "i"(limit), [then] "r"(then)
      : "cc");
  return otherwise;
#else
  (void)value;
  return below ? then : otherwise;
#endif
}

// value >= limit ? then : otherwise, likewise
inline uint32_t select_not_below(uint32_t value, uint64_t limit, uint32_t then, uint32_t otherwise) {
#if defined(__x86_64__)
  asm("cmpq %[limit], %[value]\n\tcmovae %[then], %[result]"
      : [result] "+r"(otherwise)
      : [value] "r"((uint64_t)value), [limit] "r"(limit), [then] "r"(then)
      : "cc");
  return otherwise;
#else
  return value >= limit ? then : otherwise;
#endif
}

// The same where nothing has to be checked but the contexts' liveness: contexts in range, a state
// in [2^23, 2^31) and at least two bytes a symbol and two more in the stream.  The state is the
// serial chain: bucket, entry load, multiply, refill.  The refill takes no branch (its outcome is
// as random as the stream) and no count either: the states after zero, one and two bytes are all
// made and two compares pick one, which is four cycles of the chain where a count and two shifts
// are eight.  Returns false on a context that is not live.
template <class ContextFn>
bool walk_fast(const SymbolTables &t, const uint8_t *stream, ContextFn context, uint32_t count, Position &at, uint16_t *out) {
  const uint8_t *entries = reinterpret_cast<const uint8_t *>(t.entries());
  constexpr uint32_t kPitchBits = SymbolTables::kBucketBits + 3;  // of a context's entries, in bytes
  uint32_t x = at.state;
  const uint8_t *ip = stream + at.ip;
  for (uint32_t i = 0; i < count; ++i) {
    const uint32_t c = context(i), slot = x & (kTotal - 1);
    uint16_t two;
    std::memcpy(&two, ip, 2);
    two = __builtin_bswap16(two);
    // (three loads of the entry's fields side by side, not one that the chain then shifts apart)
    const uint8_t *of_context = entries + ((size_t)c << kPitchBits);
    asm("" : "+r"(of_context));  // (made ahead of the chain: the bucket's offset goes into the loads' address)
    const auto *at_bucket = reinterpret_cast<const SymbolTables::Entry *>(
        of_context + ((x >> (SymbolTables::kBucketShift - 3)) & ((1u << kPitchBits) - 8)));
    uint32_t freq = at_bucket->freq, rel = slot - at_bucket->start, symbol = at_bucket->symbol;
    if (__builtin_expect(rel >= freq, 0)) {
      if (!t.live(c)) return false;
      const SymbolTables::Entry e = t.find(c, slot, symbol);
      freq = e.freq, rel = slot - e.start, symbol = e.symbol;
    }
    out[i] = (uint16_t)symbol;
    x = freq * (x >> kScaleBits) + rel;
    const uint32_t one_more = (x << 8) | (two >> 8), two_more = (x << 16) | two;
    const bool low = x < kLow, lower = x < (kLow >> 8);
    ip += (size_t)low + (size_t)lower;
    x = select_below<(kLow >> 8)>(lower, x, two_more, select_below<kLow>(low, x, one_more, x));
  }
  at.state = x;
  at.ip = (size_t)(ip - stream);
  return true;
}

// One forward pass over a stream, in runs: `context.run(i, most)` gives the length of the next run
// (from symbol i, at most `most`) and `context.of(k)` the model row of its k-th symbol;
// `mark(i, state, ip)` is called before symbol i where `mark.next()` says so.
struct NoProgress {
  void reached(uint64_t) {}
  bool wait_for(uint64_t) { return true; }
};
template <class Contexts, class Mark, class Progress = NoProgress>
Walk walk_stream(const uint8_t *stream, size_t bytes, uint64_t n, const SymbolTables &t, Contexts contexts, Mark &mark,
                 uint16_t *out, Progress progress = Progress{}) {
  Position at{0, 4};
  if (!read_head(stream, bytes, at.state)) return Walk::bad_head;
  const bool in_range = contexts.in_range(t.nctx());
  for (uint64_t i = 0; i < n;) {
    if (i == mark.next()) mark(i, at.state, at.ip);
    // (towards the stream's end shorter runs, so that only its last symbols are walked with every check)
    const size_t room = bytes - at.ip > 130 ? (bytes - at.ip - 2) / 2 : 64;
    const uint32_t count = contexts.run(i, (uint32_t)std::min<uint64_t>({n - i, mark.next() - i, room, 1u << 16}));
    if (!progress.wait_for(i + count)) return Walk::abandoned;
    auto context = contexts.of();
    if (in_range && at.state < 0x80000000u && at.ip + 2 * (size_t)count + 2 <= bytes) {
      if (!walk_fast(t, stream, context, count, at, out + i)) return Walk::dead_context;
    } else {
      const Walk w = walk_checked(t, stream, bytes, context, count, at, out + i);
      if (w != Walk::ok) return w;
    }
    i += count;
    progress.reached(i);
  }
  return (at.ip == bytes && at.state == kLow) ? Walk::ok : Walk::bad_tail;
}

struct NoMark {
  uint64_t next() const { return std::numeric_limits<uint64_t>::max(); }
  void operator()(uint64_t, uint32_t, size_t) {}
};

struct StrideMark {
  uint32_t stride;
  uint32_t *states, *offsets;
  uint64_t at = 0;
  size_t k = 0;
  uint64_t next() const { return at; }
  void operator()(uint64_t, uint32_t state, size_t ip) {
    states[k] = state;
    offsets[k] = (uint32_t)ip;
    ++k;
    at += stride;
  }
};

// Row-major (row class, column class) contexts; a run stays inside a row.
struct GridContext {
  const uint8_t *rc, *cc;
  uint32_t rows, cols, nc;
  uint32_t row = 0, col = 0;  // where the next run begins
  uint32_t base = 0;          // of the current run: its row's first context ...
  const uint8_t *classes = nullptr;  // ... and its columns' classes
  bool in_range(uint32_t nctx) const {
    uint32_t top_row = 0, top_col = 0;
    for (uint32_t r = 0; r < rows; ++r) top_row = std::max<uint32_t>(top_row, rc[r]);
    for (uint32_t c = 0; c < cols; ++c) top_col = std::max<uint32_t>(top_col, cc[c]);
    return top_row * nc + top_col < nctx;
  }
  uint32_t run(uint64_t, uint32_t most) {
    base = (uint32_t)rc[row] * nc;
    classes = cc + col;
    const uint32_t count = std::min(most, cols - col);
    col += count;
    if (col == cols) col = 0, ++row;
    return count;
  }
  auto of() const {
    return [base = base, classes = classes](uint32_t k) { return base + classes[k]; };
  }
};
struct ArrayContext {
  const uint16_t *ctx;
  uint64_t n;
  const uint16_t *at = nullptr;
  bool in_range(uint32_t nctx) const {
    uint32_t top = 0;
    for (uint64_t i = 0; i < n; ++i) top = std::max<uint32_t>(top, ctx[i]);
    return top < nctx;
  }
  uint32_t run(uint64_t i, uint32_t most) {
    at = ctx + i;
    return most;
  }
  auto of() const {
    return [at = at](uint32_t k) { return (uint32_t)at[k]; };
  }
};

// ---- frequency normalisation: largest remainders, deterministic ties ----
// (GCR/bitexact_context_ans.cpp:17-67)
bool normalize_row(const uint64_t *count, uint32_t vocab, uint32_t *out) {
  uint64_t total = 0;
  for (uint32_t s = 0; s < vocab; ++s) total += count[s];
  if (!total) return false;
  struct Item {
    uint64_t rem;
    uint32_t sym;
  };
  std::vector<Item> items;
  int64_t sum = 0;
  for (uint32_t s = 0; s < vocab; ++s) {
    if (!count[s]) {
      out[s] = 0;
      continue;
    }
    const uint64_t scaled = count[s] << kScaleBits;
    const uint32_t f = std::max<uint32_t>(1u, (uint32_t)(scaled / total));
    out[s] = f;
    sum += f;
    items.push_back({scaled % total, s});
  }
  if (sum < (int64_t)kTotal) {
    std::sort(items.begin(), items.end(),
              [](const Item &a, const Item &b) { return a.rem != b.rem ? a.rem > b.rem : a.sym < b.sym; });
    const uint32_t deficit = kTotal - (uint32_t)sum;
    for (uint32_t j = 0; j < deficit; ++j) ++out[items[j % items.size()].sym];
  } else if (sum > (int64_t)kTotal) {
    std::sort(items.begin(), items.end(),
              [](const Item &a, const Item &b) { return a.rem != b.rem ? a.rem < b.rem : a.sym > b.sym; });
    uint32_t excess = (uint32_t)sum - kTotal;
    for (size_t j = 0; excess; j = (j + 1) % items.size())
      if (out[items[j].sym] > 1) {
        --out[items[j].sym];
        --excess;
      }
  }
  return true;
}

// ---- encoder: symbols are pushed last-to-first so decoding runs forward ----
// (GCR/bitexact_context_ans.cpp:84-108)
//
// The state is a serial chain here too: emit zero to two bytes (the states after each are made
// and two compares pick one, no branch), divide by the symbol's frequency, recombine.  The
// division is the upper half of a product with m = floor((2^64 - 1) / f) + 1: m f = 2^64 + e with
// 0 <= e < f <= 2^16, so for x < 2^31 the error x e / (f 2^64) stays below 1 / f and the quotient is
// exact.  f = 1 would need m = 2^64; with 2^64 - 1 the quotient is x - 1 (x > 0), the remainder 1,
// and the new state 65535 short, which that symbol's bias makes up for.
// 2.6 ns a symbol where the divide instruction and the byte-wise loop took 5.6.
struct EncodeCell {
  uint64_t inverse;
  uint32_t freq, bias;  // freq 0: the symbol does not occur
};

// Writes the stream downwards from `end`; returns its first byte, or null for a symbol of frequency 0
// or when fewer than 2 n + 8 bytes are there.  value(i), context(i): i falls from n - 1 to 0.
template <class CellFn>
uint8_t *encode_stream(uint64_t n, CellFn cell_of, uint8_t *begin, uint8_t *end) {
  if ((uint64_t)(end - begin) < 2 * n + 8) return nullptr;
  uint8_t *p = end;
  uint32_t x = kLow, dead = 0;
  for (uint64_t i = n; i-- > 0;) {
    const EncodeCell &e = cell_of(i);
    const uint32_t f = e.freq;
    dead |= f == 0;
    const uint16_t two = __builtin_bswap16((uint16_t)x);
    std::memcpy(p - 2, &two, 2);
    // below f << 15 nothing leaves, below f << 23 one byte does (64-bit: f << 23 may pass 2^32)
    const uint64_t one_from = (uint64_t)f << 15, two_from = (uint64_t)f << 23;
    const bool one = x >= one_from, more = x >= two_from;
    p -= (size_t)one + (size_t)more;
    const uint32_t y = select_not_below(x, two_from, x >> 16, select_not_below(x, one_from, x >> 8, x));
    const uint64_t q = (uint64_t)(((unsigned __int128)y * e.inverse) >> 64);
    x = y + e.bias + (uint32_t)q * (kTotal - f);
  }
  if (dead) return nullptr;
  p -= 4;
  for (int k = 0; k < 4; ++k) p[k] = (uint8_t)(x >> (8 * k));
  return p;
}

std::vector<EncodeCell> encode_cells(const uint32_t *freq, uint32_t nctx, uint32_t vocab) {
  std::vector<EncodeCell> cells((size_t)nctx * vocab, EncodeCell{0, 0, 0});
  for (uint32_t c = 0; c < nctx; ++c) {
    uint32_t start = 0;
    for (uint32_t s = 0; s < vocab; ++s) {
      const uint32_t f = freq[(size_t)c * vocab + s];
      if (!f) continue;
      cells[(size_t)c * vocab + s] = f == 1 ? EncodeCell{~0ull, 1, start + kTotal - 1} : EncodeCell{~0ull / f + 1, f, start};
      start += f;
    }
  }
  return cells;
}

// fn(part, lo, hi) over [0, n) cut into parts, one thread each (the last on the caller's); small work in one part
template <class Fn>
void in_parts(uint64_t n, uint64_t least, uint32_t parts, Fn fn) {
  parts = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>({parts, n / std::max<uint64_t>(1, least), std::max(1u, std::thread::hardware_concurrency())}));
  struct Threads : std::vector<std::thread> {  // joined however this ends: the work is on the caller's memory
    ~Threads() {
      for (auto &t : *this) t.join();
    }
  } others;
  others.reserve(parts);
  uint32_t k = 0;
  for (; k + 1 < parts; ++k) try {
      others.emplace_back(fn, k, n * k / parts, n * (k + 1) / parts);
    } catch (const std::system_error &) {  // no thread to be had: the rest here
      break;
    }
  fn(k, n * k / parts, n);
}

// How far a walk has got, published now and then for a thread that follows it.
struct Counter {
  uint64_t *at = nullptr;  // symbols done; kGaveUp once the walk has failed
  uint64_t seen = 0;
  static constexpr uint64_t kGaveUp = std::numeric_limits<uint64_t>::max();
  void publish(uint64_t i) const { __atomic_store_n(at, i, __ATOMIC_RELEASE); }
  // false: the walk that is followed failed
  bool await(uint64_t i) {
    for (uint32_t spins = 0; seen < i; ++spins) {
      seen = __atomic_load_n(at, __ATOMIC_ACQUIRE);
      if (seen >= i) break;
      if (spins > 64) std::this_thread::yield();
    }
    return seen != kGaveUp;
  }
};

// Contexts of a residual walk that follows the walk of the main symbols: `ctx` is written while it is read,
// so its range is the main alphabet's, which the tables of that walk guarantee.
struct FollowingContext : ArrayContext {
  uint32_t step = 0;  // symbols it is allowed to ask for at once
  uint32_t run(uint64_t i, uint32_t most) { return ArrayContext::run(i, std::min(most, step)); }
  bool in_range(uint32_t nctx) const { return nctx >= 1024; }
};

// words[i] = main symbol on entry; the BF16 word of it and the i-th packed 6-bit field on return
void join6(uint16_t *words, const uint8_t *packed, uint64_t lo, uint64_t hi) {  // lo: a multiple of four
  auto word = [](uint32_t m, uint32_t r) { return (uint16_t)((m << 5) | (r & 31u) | ((r & 32u) << 10)); };
  const uint8_t *q = packed + lo / 4 * 3;
  uint64_t i = lo;
  for (; i + 4 <= hi; i += 4, q += 3) {
    const uint32_t v = (uint32_t)q[0] << 16 | (uint32_t)q[1] << 8 | q[2];
    words[i] = word(words[i], v >> 18);
    words[i + 1] = word(words[i + 1], (v >> 12) & 63);
    words[i + 2] = word(words[i + 2], (v >> 6) & 63);
    words[i + 3] = word(words[i + 3], v & 63);
  }
  for (uint32_t k = 0; i < hi; ++i, ++k) {  // the last one to three of a matrix
    uint32_t r = 0;
    for (uint32_t b = 0; b < 6; ++b) r = r << 1 | ((q[(6 * k + b) / 8] >> (7 - (6 * k + b) % 8)) & 1u);
    words[i] = word(words[i], r);
  }
}

struct BcxShape {
  uint32_t vocab, nctx;
};
inline BcxShape bcx_shape(uint32_t kind, uint32_t nr, uint32_t nc) {
  return kind ? BcxShape{64u, 1024u} : BcxShape{1024u, nr * nc};
}

// histogram + normalisation shared by the encoders; rows are counted in parts on a few threads
constexpr uint32_t kCountThreads = 4;
constexpr uint64_t kCountPart = 1u << 20;  // words worth a thread
void bcx_count_and_normalize(const uint16_t *w, uint32_t rows, uint32_t cols, const uint8_t *rc, const uint8_t *cc,
                             uint32_t nc, uint32_t kind, BcxShape sh, uint32_t *freq) {
  const size_t cells = (size_t)sh.nctx * sh.vocab;
  std::vector<uint32_t> counts(cells * kCountThreads);
  in_parts(rows, (kCountPart + cols - 1) / cols, kCountThreads, [&](uint32_t part, uint64_t lo, uint64_t hi) {
    uint32_t *h = counts.data() + part * cells;
    for (uint64_t r = lo; r < hi; ++r) {
      const uint16_t *row = w + r * cols;
      if (kind) {
        for (uint32_t c = 0; c < cols; ++c) ++h[main_symbol(row[c]) * 64 + residual_symbol(row[c])];
      } else {
        uint32_t *hr = h + (size_t)rc[r] * nc * 1024;
        for (uint32_t c = 0; c < cols; ++c) ++hr[(size_t)cc[c] * 1024 + main_symbol(row[c])];
      }
    }
  });
  std::vector<uint64_t> hist(sh.vocab);
  for (uint32_t c = 0; c < sh.nctx; ++c) {
    for (uint32_t s = 0; s < sh.vocab; ++s) {
      hist[s] = 0;
      for (uint32_t k = 0; k < kCountThreads; ++k) hist[s] += counts[k * cells + (size_t)c * sh.vocab + s];
    }
    normalize_row(hist.data(), sh.vocab, freq + (size_t)c * sh.vocab);
  }
}

// one symbol stream with the frequencies bcx_count_and_normalize gives, into [begin, end); its first byte, or null
uint8_t *bcx_encode_stream(const uint16_t *w, uint32_t rows, uint32_t cols, const uint8_t *rc, const uint8_t *cc, uint32_t nr,
                           uint32_t nc, uint32_t kind, const uint32_t *freq, uint8_t *begin, uint8_t *end) {
  const BcxShape sh = bcx_shape(kind, nr, nc);
  const std::vector<EncodeCell> cells = encode_cells(freq, sh.nctx, sh.vocab);
  const EncodeCell *e = cells.data();
  const uint64_t n = (uint64_t)rows * cols;
  if (kind)
    return encode_stream(
        n, [=](uint64_t i) -> const EncodeCell & { return e[main_symbol(w[i]) * 64 + residual_symbol(w[i])]; }, begin, end);
  // (the row's contexts, kept while its columns go by)
  uint32_t row = rows, col = 0;
  const EncodeCell *of_row = e;
  return encode_stream(
      n,
      [=](uint64_t i) mutable -> const EncodeCell & {
        if (col == 0) {
          of_row = e + (size_t)rc[--row] * nc * 1024;
          col = cols;
        }
        --col;
        return of_row[(size_t)cc[col] * 1024 + main_symbol(w[i])];
      },
      begin, end);
}

int bcx_decode_any(const uint8_t *stream, size_t bytes, uint64_t n, uint32_t rows, uint32_t cols,
                   const uint8_t *rc, const uint8_t *cc, uint32_t nr, uint32_t nc, uint32_t kind,
                   const uint16_t *resctx, const uint32_t *freq, uint16_t *out) {
  if (!stream || !rc || !cc || !freq || !out || !cols || !rows || kind > 1 || !nr || !nc || nr > 64 ||
      nc > 16 || (kind && !resctx) || n != (uint64_t)rows * cols)
    return 1;
  const BcxShape sh = bcx_shape(kind, nr, nc);
  SymbolTables t;
  // the reference bounds each frequency by the room left in its row
  if (t.build(freq, sh.nctx, sh.vocab) != SymbolTables::Check::ok) return 2;
  NoMark none;
  Walk w = kind ? walk_stream(stream, bytes, n, t, ArrayContext{resctx, n}, none, out)
                : walk_stream(stream, bytes, n, t, GridContext{rc, cc, rows, cols, nc}, none, out);
  return w == Walk::ok ? 0 : 2;
}

template <class Fn>
int guarded(Fn fn, int on_alloc, int on_other) {
  try {
    return fn();
  } catch (const std::bad_alloc &) {
    return on_alloc;
  } catch (...) {
    return on_other;
  }
}

}  // namespace

extern "C" {

int bcx_encode(const uint16_t *w, uint64_t n, uint32_t rows, uint32_t cols, const uint8_t *rc,
               const uint8_t *cc, uint32_t nr, uint32_t nc, uint32_t kind, uint32_t *freq, uint8_t **stream,
               size_t *stream_n) {
  return guarded(
      [&]() -> int {
        if (!w || !rc || !cc || !freq || !stream || !stream_n || n != (uint64_t)rows * cols) return 1;
        const std::unique_ptr<uint8_t[]> bytes(new uint8_t[2 * n + 8]);
        uint8_t *end = bytes.get() + 2 * n + 8;
        bcx_count_and_normalize(w, rows, cols, rc, cc, nc, kind, bcx_shape(kind, nr, nc), freq);
        const uint8_t *at = bcx_encode_stream(w, rows, cols, rc, cc, nr, nc, kind, freq, bytes.get(), end);
        if (!at) return 3;
        auto *p = (uint8_t *)std::malloc((size_t)(end - at));
        if (!p) return 2;
        std::memcpy(p, at, (size_t)(end - at));
        *stream = p;
        *stream_n = (size_t)(end - at);
        return 0;
      },
      3, 3);
}

int grf_bctx_encode(const uint16_t *w, uint32_t rows, uint32_t cols, const uint8_t *rc, const uint8_t *cc, uint32_t nr,
                    uint32_t nc, uint32_t kind, const uint32_t *freq, uint8_t *buffer, size_t buffer_bytes, size_t *begin) {
  return guarded(
      [&]() -> int {
        if (!w || !rc || !cc || !freq || !buffer || !begin || !rows || !cols) return 1;
        const uint8_t *at = bcx_encode_stream(w, rows, cols, rc, cc, nr, nc, kind, freq, buffer, buffer + buffer_bytes);
        if (!at) return 3;
        *begin = (size_t)(at - buffer);
        return 0;
      },
      3, 3);
}

int grf_bctx_sums(const uint16_t *w, uint32_t rows, uint32_t cols, uint64_t *row_sum, uint64_t *col_sum) {
  return guarded(
      [&]() -> int {
        if (!w || !row_sum || !col_sum) return 1;
        std::fill(col_sum, col_sum + cols, 0);
        std::vector<uint64_t> columns((size_t)cols * kCountThreads, 0);
        std::vector<uint32_t> partial((size_t)cols * kCountThreads, 0);  // of at most 65536 rows at a time: 16 + 15 bits
        in_parts(rows, (kCountPart + cols - 1) / cols, kCountThreads, [&](uint32_t part, uint64_t lo, uint64_t hi) {
          uint64_t *total = columns.data() + (size_t)part * cols;
          uint32_t *some = partial.data() + (size_t)part * cols;
          for (uint64_t r = lo; r < hi; ++r) {
            const uint16_t *row = w + r * cols;
            uint64_t sum = 0;
            for (uint32_t c0 = 0; c0 < cols; c0 += 65536) {
              uint32_t run = 0;
              for (uint32_t c = c0, end = std::min(cols, c0 + 65536); c < end; ++c) {
                const uint32_t v = row[c] & 0x7FFFu;
                run += v;
                some[c] += v;
              }
              sum += run;
            }
            row_sum[r] = sum;
            if ((r - lo) % 65536 == 65535 || r + 1 == hi)
              for (uint32_t c = 0; c < cols; ++c) total[c] += some[c], some[c] = 0;
          }
        });
        for (uint32_t k = 0; k < kCountThreads; ++k)
          for (uint32_t c = 0; c < cols; ++c) col_sum[c] += columns[(size_t)k * cols + c];
        return 0;
      },
      3, 3);
}

int bcx_frequencies(const uint16_t *w, uint64_t n, uint32_t rows, uint32_t cols, const uint8_t *rc,
                    const uint8_t *cc, uint32_t nr, uint32_t nc, uint32_t kind, uint32_t *freq) {
  return guarded(
      [&]() -> int {
        if (!w || !rc || !cc || !freq || n != (uint64_t)rows * cols) return 1;
        bcx_count_and_normalize(w, rows, cols, rc, cc, nc, kind, bcx_shape(kind, nr, nc), freq);
        return 0;
      },
      3, 3);
}

int bcx_decode(const uint8_t *stream, size_t bytes, uint64_t n, uint32_t rows, uint32_t cols,
               const uint8_t *rc, const uint8_t *cc, uint32_t nr, uint32_t nc, uint32_t kind,
               const uint16_t *resctx, const uint32_t *freq, uint16_t *out) {
  return guarded([&] { return bcx_decode_any(stream, bytes, n, rows, cols, rc, cc, nr, nc, kind, resctx, freq, out); },
                 3, 3);
}

// Same lookup structure serves both entry points; the reference keeps two
// decoders whose results are required to be identical.
int bcx_decode_compact(const uint8_t *stream, size_t bytes, uint64_t n, uint32_t rows, uint32_t cols,
                       const uint8_t *rc, const uint8_t *cc, uint32_t nr, uint32_t nc, uint32_t kind,
                       const uint16_t *resctx, const uint32_t *freq, uint16_t *out) {
  return guarded([&] { return bcx_decode_any(stream, bytes, n, rows, cols, rc, cc, nr, nc, kind, resctx, freq, out); },
                 3, 3);
}

void bcx_free(void *p) { std::free(p); }

// 6-bit residuals, most significant bit first; four symbols fill three bytes.
int bcx_pack6(const uint16_t *w, uint64_t n, uint8_t **out, size_t *bytes) {
  if (!w || !out || !bytes) return 1;
  const size_t z = (size_t)((n * 6 + 7) / 8);
  auto *p = (uint8_t *)std::calloc(z ? z : 1, 1);
  if (!p) return 2;
  uint64_t i = 0;
  uint8_t *q = p;
  for (; i + 4 <= n; i += 4, q += 3) {
    const uint32_t v = residual_symbol(w[i]) << 18 | residual_symbol(w[i + 1]) << 12 |
                       residual_symbol(w[i + 2]) << 6 | residual_symbol(w[i + 3]);
    q[0] = (uint8_t)(v >> 16);
    q[1] = (uint8_t)(v >> 8);
    q[2] = (uint8_t)v;
  }
  if (i < n) {
    uint32_t v = 0;
    const unsigned left = (unsigned)(n - i);
    for (unsigned k = 0; k < left; ++k) v |= residual_symbol(w[i + k]) << (18 - 6 * k);
    const unsigned nb = (left * 6 + 7) / 8;
    for (unsigned k = 0; k < nb; ++k) q[k] = (uint8_t)(v >> (16 - 8 * k));
  }
  *out = p;
  *bytes = z;
  return 0;
}

int bcx_unpack6(const uint8_t *in, size_t bytes, uint64_t n, uint16_t *out) {
  if (!in || !out || bytes != (n * 6 + 7) / 8) return 1;
  const unsigned tail_bits = (unsigned)(n * 6 % 8);
  if (tail_bits && (in[bytes - 1] & ((1u << (8 - tail_bits)) - 1))) return 2;
  uint64_t i = 0;
  const uint8_t *q = in;
  for (; i + 4 <= n; i += 4, q += 3) {
    const uint32_t v = (uint32_t)q[0] << 16 | (uint32_t)q[1] << 8 | q[2];
    out[i] = (uint16_t)(v >> 18);
    out[i + 1] = (uint16_t)((v >> 12) & 63);
    out[i + 2] = (uint16_t)((v >> 6) & 63);
    out[i + 3] = (uint16_t)(v & 63);
  }
  if (i < n) {
    const unsigned left = (unsigned)(n - i), nb = (left * 6 + 7) / 8;
    uint32_t v = 0;
    for (unsigned k = 0; k < nb; ++k) v |= (uint32_t)q[k] << (16 - 8 * k);
    for (unsigned k = 0; k < left; ++k) out[i + k] = (uint16_t)((v >> (18 - 6 * k)) & 63);
  }
  return 0;
}

int bcx_checkpoint(const uint8_t *stream, size_t stream_bytes, uint64_t n, uint32_t rows, uint32_t cols,
                   const uint8_t *rc, const uint8_t *cc, uint32_t nr, uint32_t nc, uint32_t kind,
                   const uint16_t *resctx, const uint32_t *freq, uint32_t stride, uint32_t *states,
                   uint32_t *offsets, uint16_t *out) {
  return guarded(
      [&]() -> int {
        if (!stream || !rc || !cc || !freq || !states || !offsets || !out || !rows || !cols || !nr || !nc ||
            nr > 64 || nc > 16 || !stride || kind > 1 || (kind == 1 && !resctx) ||
            n != (uint64_t)rows * (uint64_t)cols || !n || stream_bytes < 4 ||
            stream_bytes > std::numeric_limits<uint32_t>::max())
          return 1;
        const BcxShape sh = bcx_shape(kind, nr, nc);
        if (std::any_of(rc, rc + rows, [&](uint8_t v) { return v >= nr; })) return 1;
        if (std::any_of(cc, cc + cols, [&](uint8_t v) { return v >= nc; })) return 1;
        if (kind)
          for (uint64_t i = 0; i < n; ++i)
            if (resctx[i] >= sh.nctx) return 1;
        SymbolTables t;
        if (t.build(freq, sh.nctx, sh.vocab) != SymbolTables::Check::ok) return 2;
        const size_t count = (size_t)((n - 1) / stride + 1);
        // Work on private buffers: the caller's arrays change only on success.
        std::vector<uint32_t> st(count), of(count);
        std::vector<uint16_t> sym((size_t)n);
        StrideMark mark{stride, st.data(), of.data()};
        Walk w = kind ? walk_stream(stream, stream_bytes, n, t, ArrayContext{resctx, n}, mark, sym.data())
                      : walk_stream(stream, stream_bytes, n, t, GridContext{rc, cc, rows, cols, nc}, mark, sym.data());
        switch (w) {
          case Walk::ok:
            break;
          case Walk::bad_context:
          case Walk::dead_context:
          case Walk::bad_symbol:
            return 2;
          default:
            return 3;
        }
        std::copy(st.begin(), st.end(), states);
        std::copy(of.begin(), of.end(), offsets);
        std::copy(sym.begin(), sym.end(), out);
        return 0;
      },
      5, 6);
}

int grf_bctx_words(const uint8_t *stream, size_t stream_bytes, uint32_t rows, uint32_t cols, const uint8_t *rc,
                   const uint8_t *cc, uint32_t nr, uint32_t nc, const uint32_t *freq, uint32_t stride, uint32_t *states,
                   uint32_t *offsets, const uint8_t *residual, size_t residual_bytes, const uint32_t *residual_freq,
                   uint16_t *words, uint64_t *progress) {
  // Two chains: the main symbols, and what makes words of them -- the packed fields, or the
  // conditional stream, whose contexts they are.  The second follows the first a few thousand
  // symbols behind on a thread of its own (small matrices: afterwards), and `progress` tells a
  // third, the caller's, how many words are done (to hash them meanwhile).
  constexpr uint64_t kThreadFrom = 1u << 18, kStep = 1u << 13;
  Counter main_done{}, words_done{progress};
  uint64_t main_at = 0, own_at = 0;
  if (!progress) words_done.at = &own_at;
  main_done.at = &main_at;
  const int status = guarded(
      [&]() -> int {
        if (!stream || !rc || !cc || !freq || !rows || !cols || !nr || !nc || nr > 64 || nc > 16 || !residual || !words ||
            stream_bytes < 4)
          return 1;
        // (only the index has to hold its offsets in 32 bits)
        if (stride && (!states || !offsets || stream_bytes > std::numeric_limits<uint32_t>::max())) return 1;
        if (std::any_of(rc, rc + rows, [&](uint8_t v) { return v >= nr; })) return 1;
        if (std::any_of(cc, cc + cols, [&](uint8_t v) { return v >= nc; })) return 1;
        const uint64_t n = (uint64_t)rows * cols;
        if (!residual_freq) {
          if (residual_bytes != (n * 6 + 7) / 8) return 33;
          const unsigned tail_bits = (unsigned)(n * 6 % 8);
          if (tail_bits && (residual[residual_bytes - 1] & ((1u << (8 - tail_bits)) - 1))) return 33;
        }
        SymbolTables main_tables, residual_tables;
        if (main_tables.build(freq, nr * nc, 1024) != SymbolTables::Check::ok) return 2;
        if (residual_freq && residual_tables.build(residual_freq, 1024, 64) != SymbolTables::Check::ok) return 18;
        std::vector<uint16_t> fields(residual_freq ? (size_t)n : 0);

        // the second chain; a failed walk before it ends it too
        int second = 0;
        auto follow = [&] {
          Counter behind = main_done;
          if (!residual_freq) {
            for (uint64_t i = 0; i < n;) {
              const uint64_t to = std::min(n, i + kStep);
              if (!behind.await(to)) return words_done.publish(Counter::kGaveUp);
              join6(words, residual, i, to);
              words_done.publish(i = to);
            }
            return;
          }
          struct Behind {
            Counter *main, *done;
            uint16_t *words;
            const uint16_t *fields;
            uint64_t joined = 0, next = 0;
            bool wait_for(uint64_t i) { return main->await(i); }
            void reached(uint64_t i) {
              for (; joined < i; ++joined) {
                const uint32_t r = fields[joined];
                words[joined] = (uint16_t)((words[joined] << 5) | (r & 31u) | ((r & 32u) << 10));
              }
              if (i >= next) done->publish(i), next = i + kStep;
            }
          };
          NoMark unmarked;
          FollowingContext contexts;
          contexts.ctx = words;
          contexts.n = n;
          contexts.step = kStep;
          Behind progress_behind{&behind, &words_done, words, fields.data()};
          const Walk w = walk_stream(residual, residual_bytes, n, residual_tables, contexts, unmarked, fields.data(),
                                     progress_behind);
          second = w == Walk::ok || w == Walk::abandoned ? 0 : residual_bytes < 4 ? 17 : w == Walk::dead_context ? 18 : 19;
          words_done.publish(w == Walk::ok ? n : Counter::kGaveUp);
        };

        struct Ahead {
          Counter *done;
          uint64_t next = 0;
          bool wait_for(uint64_t) { return true; }
          void reached(uint64_t i) {
            if (i >= next) done->publish(i), next = i + kStep;
          }
        } ahead{&main_done};
        std::thread other;
        if (n >= kThreadFrom) try {
            other = std::thread(follow);
          } catch (const std::system_error &) {  // (no thread to be had: afterwards, then)
          }
        NoMark unmarked;
        StrideMark marked{stride, states, offsets};
        const GridContext grid{rc, cc, rows, cols, nc};
        const Walk w = stride ? walk_stream(stream, stream_bytes, n, main_tables, grid, marked, words, ahead)
                              : walk_stream(stream, stream_bytes, n, main_tables, grid, unmarked, words, ahead);
        // (a stream that ends in the wrong place is found out after its last symbol)
        main_done.publish(w == Walk::ok ? n : Counter::kGaveUp);
        if (other.joinable()) other.join();
        else follow();
        if (w != Walk::ok) return w == Walk::dead_context || w == Walk::bad_context ? 2 : 3;
        return second;
      },
      5, 6);
  if (status) words_done.publish(Counter::kGaveUp);
  return status;
}

int grf_sparse_tables(const uint32_t *freq, uint32_t nctx, uint32_t vocab, uint32_t shift, const uint32_t *image,
                      uint32_t tabn, uint8_t *lut, uint64_t *tab) {
  if (!freq || !image || !lut || !tab || !nctx || !vocab || shift > 16 || !tabn || tabn > 255) return 1;
  const uint32_t nb = kTotal >> shift;
  std::memset(lut, 0, (size_t)nctx * nb);
  std::memset(tab, 0, (size_t)nctx * (tabn + 1) * 8);
  std::vector<uint32_t> ends(tabn);
  for (uint32_t c = 0; c < nctx; ++c) {
    const uint32_t *f = freq + (size_t)c * vocab;
    uint8_t *q = lut + (size_t)c * nb;
    uint64_t *e = tab + (size_t)c * (tabn + 1);
    uint32_t k = 0, start = 0;
    for (uint32_t s = 0; s < vocab; ++s) {
      if (!f[s]) continue;
      if (k == tabn || f[s] > kTotal - start) return 2;
      e[k] = (uint64_t)image[s] << 32 | (f[s] & 0xFFFFu) << 16 | start;
      ends[k++] = start += f[s];
    }
    if (!k) continue;
    if (start != kTotal) return 2;
    uint32_t i = 0;
    for (uint32_t b = 0; b < nb; ++b) {
      const uint32_t lo = b << shift, hi = lo + (1u << shift);
      while (ends[i] <= lo) ++i;
      uint32_t best = i, most = std::min(ends[i], hi) - lo;
      for (uint32_t j = i; ends[j] < hi; ++j) {  // the symbols that begin inside the bucket
        const uint32_t held = std::min(ends[j + 1], hi) - ends[j];
        if (held > most) best = j + 1, most = held;
      }
      q[b] = (uint8_t)best;
    }
  }
  return 0;
}

int grf_order_records(const uint8_t *src, uint32_t rows, uint32_t spr, uint32_t per_segment, uint32_t record_bytes,
                      uint32_t block, const uint32_t *position, uint32_t held, uint8_t *dst) {
  if (!src || !dst || !position || !block || record_bytes % 4 || !record_bytes || record_bytes > 32) return 1;
  for (uint32_t row = 0; row < rows; ++row)
    if (position[row] >= held) return 1;
  auto move = [&](auto size) {
    constexpr size_t n = decltype(size)::value;
    for (uint32_t row = 0; row < rows; ++row) {
      const uint32_t q = position[row], within = q % block;
      const uint8_t *from = src + (size_t)row * spr * per_segment * n;
      for (uint32_t s = 0; s < spr; ++s)
        for (uint32_t t = 0; t < per_segment; ++t, from += n)
          std::memcpy(dst + ((((size_t)(q / block) * per_segment + t) * spr + s) * block + within) * n, from, n);
    }
  };
  switch (record_bytes) {
    case 12: move(std::integral_constant<size_t, 12>{}); break;
    case 16: move(std::integral_constant<size_t, 16>{}); break;
    case 20: move(std::integral_constant<size_t, 20>{}); break;
    default: return 1;
  }
  return 0;
}

int grf_unit_pieces(const uint32_t *offsets, uint32_t rows, uint32_t spr, const uint32_t *row_order, uint32_t lanes,
                    uint32_t together, uint32_t *most) {
  if (!offsets || !row_order || !most || !spr || !lanes || !together) return 1;
  const uint32_t slabs = (spr + lanes - 1) / lanes;
  try {
    // per slab, the units of the last `together` rows (the slots before the first are empty) and their sum
    const uint32_t empty = grf::piece_units(false, 0u, 0u);
    std::vector<uint32_t> units((size_t)together * slabs, empty), sum(slabs, together * empty);
    uint32_t top = together * empty;
    for (uint32_t i = 0, slot = 0; i < rows; ++i, slot = slot + 1 == together ? 0 : slot + 1) {
      if (row_order[i] >= rows) return 1;
      const uint32_t *at = offsets + (size_t)row_order[i] * spr;
      uint32_t *oldest = units.data() + (size_t)slot * slabs;
      for (uint32_t b = 0; b < slabs; ++b) {
        const uint32_t first = at[b * lanes], last = at[std::min(spr, (b + 1) * lanes)];
        const uint32_t n = grf::piece_units(true, first, last);
        sum[b] += n - oldest[b];
        oldest[b] = n;
        top = std::max(top, sum[b]);
      }
    }
    *most = top;
  } catch (...) {
    return 3;
  }
  return 0;
}

// 10-bit main symbols + 6-bit residuals -> BF16 words (no reference counterpart:
// the reference recombines in numpy, GCR/bitexact_context_codec.py:426).
int grf_bctx_join(const uint16_t *main_sym, const uint16_t *res_sym, uint64_t n, uint16_t *out) {
  if (!main_sym || !res_sym || !out) return 1;
  for (uint64_t i = 0; i < n; ++i) {
    const uint32_t m = main_sym[i], r = res_sym[i];
    if (m > 1023u || r > 63u) return 2;
    out[i] = (uint16_t)((m << 5) | (r & 31u) | ((r >> 5) << 15));
  }
  return 0;
}

// ---------------------------------------------------------------- PPCX
int p_encode(const uint16_t *v, const uint16_t *cx, uint64_t n, uint32_t nc, uint32_t vocab, uint32_t **freqp,
             uint8_t **streamp, size_t *sn) {
  return guarded(
      [&]() -> int {
        if (!v || !cx || !n || n > 100000000u || !nc || !vocab || vocab > kTotal || !freqp || !streamp || !sn)
          return 1;
        *freqp = nullptr;
        *streamp = nullptr;
        *sn = 0;
        const size_t cells = (size_t)nc * vocab;
        std::vector<uint64_t> hist(cells);
        for (uint64_t i = 0; i < n; ++i) {
          if (cx[i] >= nc || v[i] >= vocab) return 2;
          ++hist[(size_t)cx[i] * vocab + v[i]];
        }
        std::vector<uint32_t> freq(cells);
        for (uint32_t c = 0; c < nc; ++c) normalize_row(hist.data() + (size_t)c * vocab, vocab, freq.data() + (size_t)c * vocab);
        const std::unique_ptr<uint8_t[]> bytes(new uint8_t[2 * n + 8]);
        uint8_t *end = bytes.get() + 2 * n + 8;
        const std::vector<EncodeCell> table = encode_cells(freq.data(), nc, vocab);
        const uint8_t *at = encode_stream(
            n, [&](uint64_t i) -> const EncodeCell & { return table[(size_t)cx[i] * vocab + v[i]]; }, bytes.get(),
            end);
        if (!at) return 3;
        const size_t size = (size_t)(end - at);
        auto *fp = (uint32_t *)std::malloc(cells * sizeof(uint32_t));
        auto *sp = (uint8_t *)std::malloc(size);
        if (!fp || !sp) {
          std::free(fp);
          std::free(sp);
          return 4;
        }
        std::memcpy(fp, freq.data(), cells * sizeof(uint32_t));
        std::memcpy(sp, at, size);
        *freqp = fp;
        *streamp = sp;
        *sn = size;
        return 0;
      },
      5, 5);
}

// The stream that p_encode would give with the frequencies it is given, one thread, for symbols that were decoded with them.
int ppcx_encode_given(const uint16_t *v, const uint16_t *cx, uint64_t n, uint32_t nc, uint32_t vocab, const uint32_t *freq,
                      uint8_t **streamp, size_t *sn) {
  return guarded(
      [&]() -> int {
        if (!v || !cx || !n || n > 100000000u || !nc || !vocab || vocab > kTotal || !freq || !streamp || !sn) return 1;
        for (uint64_t i = 0; i < n; ++i)
          if (cx[i] >= nc || v[i] >= vocab || !freq[(size_t)cx[i] * vocab + v[i]]) return 2;
        const std::unique_ptr<uint8_t[]> bytes(new uint8_t[2 * n + 8]);
        uint8_t *end = bytes.get() + 2 * n + 8;
        const std::vector<EncodeCell> table = encode_cells(freq, nc, vocab);
        const uint8_t *at = encode_stream(
            n, [&](uint64_t i) -> const EncodeCell & { return table[(size_t)cx[i] * vocab + v[i]]; }, bytes.get(), end);
        if (!at) return 3;
        const size_t size = (size_t)(end - at);
        auto *sp = (uint8_t *)std::malloc(size);
        if (!sp) return 4;
        std::memcpy(sp, at, size);
        *streamp = sp, *sn = size;
        return 0;
      },
      5, 5);
}

// Status categories follow GCR/bitexact_predictive_ans.cpp:11 (1 arguments,
// 2 initial state, 3 table row overflow, 4 row does not sum to the total,
// 5 context out of range, 8 stream exhausted, 9 terminal state/length).
int p_decode(const uint8_t *st, size_t bytes, uint64_t n, const uint16_t *cx, uint32_t nc, uint32_t vocab,
             const uint32_t *f, uint16_t *out) {
  return guarded(
      [&]() -> int {
        if (!st || bytes < 4 || !cx || !f || !out || !n || n > 100000000u || !nc || !vocab || vocab > kTotal)
          return 1;
        uint32_t head;
        if (!read_head(st, bytes, head)) return 2;
        SymbolTables t;
        // a row whose sum is wrong only fails (4) when a symbol selects it
        if (t.build(f, nc, vocab, true) != SymbolTables::Check::ok) return 3;
        NoMark none;
        switch (walk_stream(st, bytes, n, t, ArrayContext{cx, n}, none, out)) {
          case Walk::ok:
            return 0;
          case Walk::bad_context:
            return 5;
          case Walk::dead_context:
            return 4;
          case Walk::overrun:
            return 8;
          case Walk::bad_head:
            return 2;
          default:
            return 9;
        }
      },
      10, 10);
}

void p_free(void *p) { std::free(p); }

static int ppcx_checkpoint_impl(const uint8_t *stream, size_t bytes, uint64_t n, const uint16_t *ctx,
                                uint32_t nctx, uint32_t vocab, const uint32_t *freq, uint32_t stride,
                                uint32_t *states, uint32_t *offsets, uint16_t *symbols) {
  return guarded(
      [&]() -> int {
        if (!stream || bytes < 4 || bytes > std::numeric_limits<uint32_t>::max() || !n || !ctx || !nctx ||
            !vocab || vocab > kTotal || !freq || !stride || !states || !offsets || !symbols || n > 100000000u)
          return 1;
        SymbolTables t;
        if (t.build(freq, nctx, vocab) != SymbolTables::Check::ok) return 2;
        const size_t count = (size_t)((n + stride - 1) / stride);
        std::vector<uint32_t> st(count), of(count);
        StrideMark mark{stride, st.data(), of.data()};
        switch (walk_stream(stream, bytes, n, t, ArrayContext{ctx, n}, mark, symbols)) {
          case Walk::ok:
            break;
          case Walk::bad_context:
            return 4;
          case Walk::dead_context:
          case Walk::bad_symbol:
            return 5;
          default:
            return 3;
        }
        std::copy(st.begin(), st.end(), states);
        std::copy(of.begin(), of.end(), offsets);
        return 0;
      },
      6, 6);
}

int ppcx_checkpoint(const uint8_t *stream, size_t bytes, uint64_t n, const uint16_t *ctx, uint32_t nctx,
                    uint32_t vocab, const uint32_t *freq, uint32_t stride, uint32_t *states, uint32_t *offsets,
                    uint16_t *symbols) {
  return ppcx_checkpoint_impl(stream, bytes, n, ctx, nctx, vocab, freq, stride, states, offsets, symbols);
}

// The reference offers a second entry point with a faster search; here both use
// the coarse-index lookup, so they are the same function.
int ppcx_checkpoint_binary(const uint8_t *stream, size_t bytes, uint64_t n, const uint16_t *ctx, uint32_t nctx,
                           uint32_t vocab, const uint32_t *freq, uint32_t stride, uint32_t *states,
                           uint32_t *offsets, uint16_t *symbols) {
  return ppcx_checkpoint_impl(stream, bytes, n, ctx, nctx, vocab, freq, stride, states, offsets, symbols);
}

}  // extern "C"
