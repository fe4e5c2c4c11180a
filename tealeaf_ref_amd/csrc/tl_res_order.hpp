// Which of its two copies of the buffers an exchange of the on-chip loops uses
// (tl_resident.hpp).  Plain C++, so that a model of the exchanges on the CPU
// takes the same rule.
//
// Halos alternate with the number of the exchange, sums with the number of the
// sum:
//  - Halos.  A wave writes a neighbour's words of exchange s + 2 after it has
//    the same neighbour's words of exchange s + 1, or, where that one exchanges
//    no halos, after a sum to which every block has added; the neighbour gave
//    either after it had read those of exchange s.
//  - Sums.  A block writes its partial of sum q + 2 after sum q + 1 has all blocks'
//    partials, and a block gives that one after it has read all of sum q.  The
//    number of the exchange would not do: an exchange of halos alone waits for
//    the neighbours only, so that blocks further apart than the exchanges
//    between two sums may still be reading the first when the second is written.
#pragma once

namespace tl {

// EVERY: every exchange of the loop carries a sum, so that the two numbers are
// one (and one register).
template <bool EVERY>
struct ResOrder {
  static constexpr bool every_sums = EVERY;
  unsigned s = 0;  // exchanges so far
  int q = 0;       // parity of the sums so far
  constexpr unsigned tag(unsigned epoch) const { return epoch + s; }
  constexpr int halos() const { return (int)(s & 1); }
  constexpr int sums() const { return EVERY ? halos() : q; }
  constexpr void next(bool sum) {
    s += 1;
    if (!EVERY) q ^= sum ? 1 : 0;
  }
};

}  // namespace tl
