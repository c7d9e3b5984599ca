"""The slots through which a short reduction's workgroups hand over their
partials: every interleaving of one writer with a reader that gives up after
few looks leaves the slot zero, and the next call's partial is its own."""

import os
import subprocess

SOURCE = r"""
#define __host__
#define __device__
#include "reduce_slots.hpp"
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <thread>
using namespace rpx;
typedef unsigned long long u64;

// One access at a time, by the thread whose turn the schedule says it is: bit i
// set for the writer.  A thread that has ended, or the schedule's end, frees the other.
static std::mutex mu;
static std::condition_variable cv;
static unsigned schedule;
static int at, length;
static bool ended[2];
static thread_local int me;
template <class F> static u64 turn(F f) {
  std::unique_lock<std::mutex> l(mu);
  cv.wait(l, [] { return at >= length || ended[1 - me] || int(schedule >> at & 1) == me; });
  const u64 r = f();
  ++at;
  cv.notify_all();
  return r;
}
static void end() {
  std::lock_guard<std::mutex> l(mu);
  ended[me] = true;
  cv.notify_all();
}
struct Turns {
  static u64 load(u64* p) { return turn([&] { return *p; }); }
  static void store(u64* p, u64 v) { turn([&] { return *p = v; }); }
  static u64 exchange(u64* p, u64 v) { return turn([&] { const u64 o = *p; *p = v; return o; }); }
  static void pause() {}
};
struct Plain {
  static u64 load(u64* p) { return *p; }
  static void store(u64* p, u64 v) { *p = v; }
  static u64 exchange(u64* p, u64 v) { const u64 o = *p; *p = v; return o; }
  static void pause() {}
};

int main() {
  long bad = 0, gave_up = 0, took = 0;
  const u64 first = 0x400921FB54442D18ull, second = 0xC005BF0A8B145769ull;
  length = 9;  // the reader's six accesses at a limit of 0, or eight at 1, beside the writer's two to four
  for (unsigned limit = 0; limit < 2; ++limit)
    for (unsigned plan = 0; plan < 1u << 9; ++plan) {
      u64 slot[2] = {0, 0}, bits = 0;
      schedule = plan, at = 0, ended[0] = ended[1] = false;
      bool got = false;
      std::thread reader([&] { me = 0; got = slot_take<Turns>(slot, limit, &bits); end(); });
      std::thread writer([&] { me = 1; slot_leave<Turns>(slot, first); end(); });
      reader.join();
      writer.join();
      ++(got ? took : gave_up);
      if (got && bits != first) bad++;
      if (slot[0] != 0 || slot[1] != 0) bad++;
      // The next call.
      got = slot_take<Plain>(slot, 3, &bits);
      if (got) bad++;
      slot_leave<Plain>(slot, second);
      if (slot[0] != 0 || slot[1] != 0) bad++;
      slot_leave<Plain>(slot, second);
      if (!slot_take<Plain>(slot, 3, &bits) || bits != second || slot[0] != 0 || slot[1] != 0) bad++;
    }
  printf("%ld wrong, %ld took, %ld gave up\n", bad, took, gave_up);
  return bad != 0 || took == 0 || gave_up == 0;
}
"""


def test_slots_are_zero_after_every_interleaving(tmp_path):
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rajaperf_amd", "csrc")
    src, exe = tmp_path / "slots.cpp", tmp_path / "slots"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", csrc, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
