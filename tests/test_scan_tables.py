"""The tables of a segmented SCAN against the look-back words that a later
single-array SCAN may keep in the same place: no entry reads as a published
status of an epoch that a program reaches (2^39 calls)."""

import os
import subprocess

SOURCE = r"""
#define __host__
#define __device__
#include "scan_words.hpp"
#include <cstdio>
#include <initializer_list>
using namespace rpx;
static unsigned long long state = 88172645463325252ull;
static unsigned long long random64() { state ^= state << 13; state ^= state >> 7; return state ^= state << 17; }
static long bad = 0;
static void check(unsigned long long word, long long what) {
  const unsigned long long epoch = word >> 24;  // the only one that could accept it
  if (epoch < 1ull << 39 && tile_status(word, epoch) != 0 && bad++ < 5) printf("%lld: epoch %llu\n", what, epoch);
}
static void entry(int64_t v) {
  check(table_entry(v), v);
  if (table_value(table_entry(v)) != v) bad++;
}
static void pair(int a, int b) {
  check((unsigned long long)segment_entry(b) << 32 | segment_entry(a), a);
  if (segment_value(segment_entry(a)) != a) bad++;
}
int main() {
  for (int64_t v : {0ll, 21000000ll, 21000010ll, 1ll << 24, (1ll << 24) + (1ll << 22), (1ll << 40) + 5, (1ll << 62) - 1}) entry(v);
  for (int a : {0, 1, 5 << 20, (1 << 22) + 1, 0x7FFFFFFF}) for (int b : {0, 1, 1 << 22, 0x7FFFFFFF}) pair(a, b);
  for (int i = 0; i < 1000000; ++i) {
    entry(int64_t(random64() >> (1 + random64() % 62)));
    pair(int(random64() >> (33 + random64() % 30)), int(random64() >> (33 + random64() % 30)));
  }
  // A published word is accepted in its own epoch only.
  for (unsigned long long e = 1; e < 1000; ++e)
    for (unsigned s = 1; s <= 2; ++s)
      if (tile_status(tile_tag(e, s) | 12345, e) != s || tile_status(tile_tag(e, s), e + 1) != 0) bad++;
  return bad != 0;
}
"""


def test_no_table_entry_is_a_status(tmp_path):
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rajaperf_amd", "csrc")
    src, exe = tmp_path / "tables.cpp", tmp_path / "tables"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", csrc, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
