// tile_hint.cpp -- host check of mx_stream::expected_rows (mx_internal.hpp), the
// row count a packed pass's GEMM tiles are chosen for, from the words that the
// plans of completed passes write. TEST PROGRAM: prints "ok" and exits 0, or
// names the first failure and exits 1.
#include <cstdio>

#include "mx_internal.hpp"

static int bad = 0;
static void expect(const char *what, int64_t got, int64_t want) {
  if (got == want) return;
  std::printf("FAIL: %s: %lld, expected %lld\n", what, (long long)got, (long long)want);
  bad = 1;
}
static uint64_t pass(int64_t B, int64_t S, int64_t rows) {
  return (uint64_t)(B * S) << 32 | (uint64_t)rows;
}

int main() {
  uint64_t words[2] = {0, 0};
  mx_stream s;
  s.note = words;
  expect("nothing seen: a sequence fills its width", s.expected_rows(1, 512), 512);
  words[1] = pass(1, 512, 20);  // a sequence of 20 in 512 columns
  expect("the same width again", s.expected_rows(1, 512), 20);
  expect("another width", s.expected_rows(1, 256), 10);
  words[0] = pass(64, 512, 16384);  // a batch, half live
  expect("a batch", s.expected_rows(32, 512), 8192);
  expect("a sequence after the batch", s.expected_rows(1, 512), 20);
  words[1] = pass(1, 19, 19);  // a sequence without padding
  expect("a sequence of its own width", s.expected_rows(1, 300), 300);
  expect("a batch after the sequence", s.expected_rows(2, 100), 100);
  words[0] = pass(64, 512, 1);
  expect("never none", s.expected_rows(2, 8), 1);
  mx_stream without;  // no pinned memory: nothing to go by
  expect("no words, a sequence", without.expected_rows(1, 77), 77);
  expect("no words, a batch", without.expected_rows(3, 7), 21);
  if (!bad) std::printf("ok\n");
  return bad;
}
