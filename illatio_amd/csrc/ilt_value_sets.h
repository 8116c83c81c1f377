// Which positions a wave of attn_values_mm_kernel asks for and which of them it adds, apart from how: they come in sets of P,
// AHEAD sets on their way at a time, and a set is added before its registers are asked for anew.  The values' cache may end
// at the last position, nposmax - 1, so a set that would reach past it lies further down instead, its end on that position;
// where there are fewer than P positions the last one stands in for what would lie past it.  So every set's loads are the
// same number of the same instructions, whatever it is: how many are on their way is known everywhere in the loop.
// (constexpr, so that a host's compiler takes it as well and a test can walk it.)
#pragma once

// The set that is asked for as positions p .. p + P - 1: slot k holds position base + at(k).
constexpr int ilt_set_base(int p, int P, int nposmax) { const int top = nposmax > P ? nposmax - P : 0; return p < top ? p : top; }
constexpr int ilt_set_at(int k, int nposmax) { return k < nposmax ? k : nposmax - 1; }
// A row of npos positions adds slot k of it where ilt_set_from(.., k) < ilt_set_left: the positions before p were other sets',
// the row's own end before npos.  (unsigned: a position before p is a large number)
constexpr unsigned ilt_set_from(int p, int base, int k) { return (unsigned)(base + k - p); }
constexpr unsigned ilt_set_left(int p, int npos) { return (unsigned)(npos > p ? npos - p : 0); }

// load(x, p) asks for the set at p, whole(x, p) adds one that all rows see whole, ends(x, p) one that may lie further down and
// inside which rows may end.  Rows end at positions npos0 - 1 .. nposmax - 1.
template <int P, int AHEAD, class Set, class Load, class Whole, class Ends>
__attribute__((always_inline)) constexpr void ilt_value_sets(Set (&x)[AHEAD], int npos0, int nposmax, Load load, Whole whole, Ends ends) {
#pragma unroll
  for (int u = 0; u < AHEAD; u++) load(x[u], P * u);
  int p = 0;
  for (; p + P * AHEAD <= npos0; p += P * AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
      whole(x[u], p + P * u);
      load(x[u], p + P * u + P * AHEAD);
    }
  }
  for (; p < nposmax; p += P * AHEAD) {
#pragma unroll
    for (int u = 0; u < AHEAD; u++) {
      const int pu = p + P * u;
      if (pu + P <= npos0) whole(x[u], pu);
      else if (pu < nposmax) ends(x[u], pu);
      if (pu + P * AHEAD < nposmax) load(x[u], pu + P * AHEAD);
    }
  }
}
