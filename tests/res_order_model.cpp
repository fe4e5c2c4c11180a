// Model of the exchanges of the on-chip loops: blocks of W waves that post and
// poll tagged words as dev::res_exchange does, with the buffers that
// tl_res_order.hpp chooses, under schedules in which single waves or whole blocks
// lag.  A poll takes a word only with the tag of its own exchange, so a word that
// is written again too early leaves its reader waiting for ever.
//
//   res_order_model        prints per loop, grid and rule the schedules that end stuck
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "tl_res_order.hpp"

constexpr int W = 3;  // waves of a block: the bottom row's, one between, the top row's

// The rule that a sum takes the copy of its exchange's number, against which the
// model is tried too.
struct ByExchange : tl::ResOrder<false> {
  constexpr int sums() const { return (int)(s & 1); }
};

struct Kind {
  bool halo, sum;
};

struct Wave {
  int at = 0, phase = 0;       // exchange, and place in it
  std::vector<int> wants;      // words to be polled: halos[i], or parts[-1 - i]
};

template <typename ORDER>
struct Model {
  int tx, ty, nb;
  std::vector<Kind> loop;
  std::vector<ORDER> order;    // of every exchange
  std::vector<unsigned> halos, parts;  // tags in the two copies
  std::vector<Wave> waves;
  std::vector<int> first, second;      // arrivals at the barriers, per block and exchange

  Model(int tx_, int ty_, std::vector<Kind> l) : tx(tx_), ty(ty_), nb(tx_ * ty_), loop(l) {
    ORDER o;
    for (Kind k : loop) {
      order.push_back(o);
      o.next(k.sum);
    }
    // a block's halo words: left and right of every wave, bottom, top
    halos.assign(2 * nb * (2 * W + 2), 0);
    parts.assign(2 * nb, 0);
    waves.resize(nb * W);
    first.assign(nb * loop.size(), 0);
    second.assign(nb * loop.size(), 0);
  }
  int side(int copy, int b, bool right, int w) const {
    return (copy * nb + b) * (2 * W + 2) + (right ? W : 0) + w;
  }
  int row(int copy, int b, bool top) const { return (copy * nb + b) * (2 * W + 2) + 2 * W + top; }
  bool finished(int i) const { return waves[i].at == (int)loop.size(); }

  // One step of wave i; whether it could make one.
  bool step(int i) {
    if (finished(i)) return false;
    Wave &v = waves[i];
    const int b = i / W, w = i % W, bx = b % tx, by = b / tx, n = v.at;
    const Kind k = loop[n];
    const unsigned tag = order[n].tag(1);
    const int hc = order[n].halos(), sc = order[n].sums();
    const size_t bar = (size_t)b * loop.size() + n;
    switch (v.phase) {
      case 0:  // post the halos
        if (k.halo) {
          if (bx > 0) halos[side(hc, b, false, w)] = tag;
          if (bx + 1 < tx) halos[side(hc, b, true, w)] = tag;
          if (w == 0 && by > 0) halos[row(hc, b, false)] = tag;
          if (w == W - 1 && by + 1 < ty) halos[row(hc, b, true)] = tag;
        }
        first[bar] += 1;
        v.phase = 1;
        return true;
      case 1:  // the first barrier, then the block's partial
        if (first[bar] < W) return false;
        if (k.sum && w == 0) parts[sc * nb + b] = tag;
        v.wants.clear();
        if (k.halo) {
          if (bx > 0) v.wants.push_back(side(hc, b - 1, true, w));
          if (bx + 1 < tx) v.wants.push_back(side(hc, b + 1, false, w));
          if (w == 0 && by > 0) v.wants.push_back(row(hc, b - tx, true));
          if (w == W - 1 && by + 1 < ty) v.wants.push_back(row(hc, b + tx, false));
        }
        // waves 1.. share the partials
        if (k.sum && w > 0)
          for (int q = w - 1; q < nb; q += W - 1) v.wants.push_back(-1 - (sc * nb + q));
        v.phase = 2;
        return true;
      case 2:  // poll: a lane reads all its words anew until each has the tag
        for (int a : v.wants)
          if ((a >= 0 ? halos[a] : parts[-1 - a]) != tag) return false;
        if (k.sum) second[bar] += 1;
        v.phase = 3;
        return true;
      default:  // the second barrier, of sums
        if (k.sum && second[bar] < W) return false;
        v.at += 1;
        v.phase = 0;
        return true;
    }
  }
  // All waves take random steps; those of `late` (a block, or a wave of it) only
  // when nothing else moves, and then one.  Whether the loop ends.
  bool run(unsigned seed, int late_block, int late_wave) {
    std::mt19937 rng(seed);
    std::vector<int> quick, slow;
    for (int i = 0; i < nb * W; ++i)
      (i / W == late_block && (late_wave < 0 || i % W == late_wave) ? slow : quick).push_back(i);
    auto any = [&](std::vector<int> &set) {
      for (size_t k = set.size(); k > 1; --k) std::swap(set[k - 1], set[rng() % k]);
      for (int i : set)
        if (step(i)) return true;
      return false;
    };
    while (any(quick) || any(slow)) {
    }
    for (int i = 0; i < nb * W; ++i)
      if (!finished(i)) return false;
    return true;
  }
};

template <typename ORDER>
void report(const char *rule, const std::string &name, int tx, int ty,
            const std::vector<Kind> &loop) {
  int runs = 0, stuck = 0;
  for (int late = 0; late < tx * ty; ++late)
    for (int wave = -1; wave < W; ++wave) {
      stuck += !Model<ORDER>(tx, ty, loop).run(7u * late + wave + 1, late, wave);
      ++runs;
    }
  std::printf("%s %s %dx%d runs %d stuck %d\n", rule, name.c_str(), tx, ty, runs, stuck);
}

int main() {
  const Kind SUM = {false, true}, HALO = {true, false}, BOTH = {true, true};
  std::vector<std::pair<std::string, std::vector<Kind>>> loops;
  std::vector<Kind> l;
  for (int n = 0; n < 6; ++n) l.insert(l.end(), {SUM, BOTH});
  loops.push_back({"cg", l});
  loops.push_back({"jacobi", std::vector<Kind>(10, BOTH)});
  l.assign(9, HALO);
  l.push_back(SUM);
  loops.push_back({"chebyshev", l});
  for (int inner : {1, 2, 3, 4, 5, 7, 9, 10}) {
    l.clear();
    for (int n = 0; n < 4; ++n) {
      l.push_back(SUM);
      l.insert(l.end(), inner, HALO);
      l.push_back(BOTH);
    }
    loops.push_back({"ppcg" + std::to_string(inner), l});
  }
  const int grids[][2] = {{1, 1}, {2, 1}, {1, 4}, {3, 4}, {12, 1}, {1, 12}};
  for (auto &lp : loops)
    for (auto &g : grids) {
      if (lp.first == "cg" || lp.first == "jacobi")
        report<tl::ResOrder<true>>("sums", lp.first, g[0], g[1], lp.second);
      else
        report<tl::ResOrder<false>>("sums", lp.first, g[0], g[1], lp.second);
      report<ByExchange>("exchanges", lp.first, g[0], g[1], lp.second);
    }
  return 0;
}
