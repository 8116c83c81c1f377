"""Which positions a prompt chunk's values are asked for and added (ilt_value_sets.h), walked by the host's compiler as the two kernels
do: no load reaches past the cache's last byte, also before any range check, and every row adds every position of its own once, in
order, from a register that holds it."""
import os
import subprocess

from illatio_amd import hip

CSRC = os.path.join(os.path.dirname(hip.__file__), "csrc")

WALK = r"""
#include "ilt_value_sets.h"
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#define CHECK(c) do { if (!(c)) { printf("%s: P %d, AHEAD %d, npos0 %d, nposmax %d, at %d\n", #c, P, AHEAD, npos0, nposmax, p); exit(1); } } while (0)

// KVD floats a position; the wave's last lane reads a position's last one
template <int P, int AHEAD> void walk(int npos0, int nposmax, long kvd) {
  struct Set { int at[P]; } x[AHEAD];                                // the position that each register holds
  for (Set& s : x) for (int& a : s.at) a = -1;
  std::vector<int> done(nposmax - npos0 + 1, 0);                     // rows of npos0 .. nposmax positions: the next one to add
  auto load = [&](Set& s, int p) {
    const long base = ilt_set_base(p, P, nposmax);
    for (int k = 0; k < P; k++) {
      const long vector = 4 * (kvd - 1) + base * kvd * 4, scalar = ilt_set_at(k, nposmax) * kvd * 4;
      CHECK(base >= 0 && scalar >= 0 && vector + scalar + 4 <= 4 * kvd * nposmax);
      s.at[k] = base + ilt_set_at(k, nposmax);
    }
  };
  auto whole = [&](const Set& s, int p) {
    CHECK(p + P <= npos0);
    for (int k = 0; k < P; k++) for (int& d : done) { CHECK(s.at[k] == p + k && d == p + k); d++; }
  };
  auto ends = [&](const Set& s, int p) {
    const int base = ilt_set_base(p, P, nposmax);
    for (int k = 0; k < P; k++)
      for (int npos = npos0; npos <= nposmax; npos++)
        if (ilt_set_from(p, base, k) < ilt_set_left(p, npos)) { int& d = done[npos - npos0]; CHECK(s.at[k] == d && d < npos); d++; }
  };
  ilt_value_sets<P, AHEAD>(x, npos0, nposmax, load, whole, ends);
  for (int p = npos0; p <= nposmax; p++) CHECK(done[p - npos0] == p);
}

int main() {
  for (int nposmax = 1; nposmax <= 400; nposmax++)
    for (int back = 0; back < 16 && back < nposmax; back++) {        // sixteen rows are of up to sixteen tokens, four of four
      walk<8, 2>(nposmax - back, nposmax, 1024);
      if (back < 4) walk<16, 3>(nposmax - back, nposmax, 64);
    }
}
"""


def test_no_load_past_the_last_position_and_every_position_added_once(tmp_path):
    (tmp_path / "walk.cpp").write_text(WALK)
    exe = str(tmp_path / "walk")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-I", CSRC, "-o", exe, str(tmp_path / "walk.cpp")])
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
