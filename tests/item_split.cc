// make_split (launch.h) over random geometries: the ranges cover every item once,
// in order, and the padded form is chosen only where its longest range, with the
// strips that it enters, is no longer than the plain split's.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "launch.h"

namespace arthip {
FastDiv make_fastdiv(uint32_t d) { return FastDiv{d, 0, 0}; }
}  // namespace arthip

using arthip::ItemSplit;

// split_begin (wino_dev.h) with plain divisions.
static int64_t begin_of(const ItemSplit& s, int64_t slot) {
  const int64_t v = slot * s.q + slot * s.r / s.slots.d;
  const int64_t strip = v / s.strip.d, len = s.strip.d - s.pad;
  return strip * len + std::max<int64_t>(v - strip * s.strip.d - s.pad, 0);
}

static int64_t longest(const ItemSplit& s, int64_t items, int64_t slots, int64_t len, int64_t fill) {
  int64_t at = 0, most = 0;
  for (int64_t k = 0; k < slots; ++k) {
    const int64_t b = begin_of(s, k), e = begin_of(s, k + 1);
    if (b != at || e < b || (s.q + 1) * slots > INT32_MAX || k * s.r > INT32_MAX) return -1;
    at = e;
    if (e > b) most = std::max(most, e - b + ((e - 1) / len - b / len) * fill);
  }
  return at == items ? most : -1;
}

int main() {
  std::mt19937 rng(5);
  auto upto = [&](int n) { return 1 + static_cast<int64_t>(rng() % n); };
  int padded = 0, shorter = 0;
  for (int i = 0; i < 20000; ++i) {
    const int64_t len = upto(i % 2 ? 70 : 1100), strips = upto(i % 3 ? 70 : 700), items = len * strips;
    const int64_t cap = i % 4 ? 256 << (rng() % 4) : 8 * upto(256);
    const int64_t slots = (std::min(cap, items) + 7) / 8 * 8, fill = rng() % 6;
    const ItemSplit s = arthip::make_split(items, slots, len, fill);
    const ItemSplit plain = arthip::make_split(items, slots, len, 0);
    const int64_t now = longest(s, items, slots, len, fill), was = longest(plain, items, slots, len, fill);
    if (now < 0 || was < 0 || now > was) {
      std::printf("%lld items in strips of %lld, %lld slots, fill %lld: longest %lld, plain %lld\n", (long long)items,
                  (long long)len, (long long)slots, (long long)fill, (long long)now, (long long)was);
      return 1;
    }
    padded += s.pad != 0;
    shorter += now < was;
  }
  std::printf("padded %d shorter %d\n", padded, shorter);
  return padded > 5000 && shorter > 5000 ? 0 : 1;
}
