"""ringattn_news.h: a round of dealt::ring_walk_kernel, with a tile that moves the references writing its word again while other waves may still be
reading it.  A model of the six waves -- their reads, writes and barriers in the order of the kernel, the words and what is found in
them by the kernel's own functions, compiled with the host compiler -- is run in orders in which any of them is late: all have to pass the same
barriers, and the waves of P V to end a round with the last version of every tile, the factors of those that moved, and the reference."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdint.h>
#include <stdio.h>
#include "ringattn_news.h"
using namespace ringattn;

constexpr int W = kNewsTiles, kWaves = W + 2, kRounds = 6;
static uint64_t state;
static int draw(int n) {
  state = state * 6364136223846793005ull + 1442695040888963407ull;
  return (int)(state >> 33) % n;
}

// The workgroup's LDS, with what stands for its contents: versions for probabilities and sums, the moving tile for factors and references.
static int news[2][W], probs[2][W], factors[2][W], reference;
static bool wants[kRounds][W][W + 1];   // does a tile want a move, by how often its exponentials have been taken before
static int fails;

struct Wave {
  int id, at, r, first, from, taken, known, passed;
  int said[W], seen[W];
  int label;   // of the barrier it waits for
  bool waits, done;
};
static Wave waves[kWaves];

static int version(int r, int tile, int taken) { return (r * W + tile) * 8 + taken + 1; }
static void look(Wave& w) { for (int i = 0; i < W; ++i) w.said[i] = news[w.r & 1][i]; }
static int bits(const Wave& w) { return news_of_round(w.said[0], w.said[1], w.said[2], w.said[3]); }
static void tell(const Wave& w, int what) {
  probs[w.r & 1][w.id] = version(w.r, w.id, w.taken);
  news[w.r & 1][w.id] = what;
}
static void wait_at(Wave& w, int which) { w.waits = true; w.label = w.r * 16 + which; }

// One access, or the way to the next barrier.
static void step(Wave& w) {
  const bool scores = w.id < W;
  switch (w.at) {
    case 0:   // the tile of the round
      w.taken = 0;
      w.passed = 0;
      if (scores) tell(w, wants[w.r][w.id][0] ? kNewsWish : 0);
      w.at = 1;
      wait_at(w, 0);
      break;
    case 1: w.from = 0; look(w); w.at = scores ? 3 : 2; break;
    case 2: for (int i = 0; i < W; ++i) w.seen[i] = probs[w.r & 1][i]; w.at = 3; break;
    case 3:
      if (w.from == W) { w.at = 9; break; }
      w.first = first_wish(bits(w), w.from);
      if (w.first >= W) { w.at = 9; break; }
      w.at = w.id == w.first ? 4 : 6;
      break;
    case 4: ++w.taken; tell(w, kNewsMoved); w.at = 5; break;
    case 5: factors[w.r & 1][w.id] = reference = w.known = version(w.r, w.id, 0); w.at = 6; break;
    case 6: w.at = 7; wait_at(w, ++w.passed); break;
    case 7:
      if (scores && w.id != w.first) w.known = reference;
      w.from = w.first + 1;
      if (w.from < W) {
        if (scores && w.id >= w.from) { ++w.taken; tell(w, wants[w.r][w.id][w.taken] ? kNewsWish : 0); }
        w.at = 8;
        wait_at(w, ++w.passed);
      } else w.at = 8;
      break;
    case 8: look(w); w.at = scores ? 3 : 2; break;
    case 9: {
      // the round as it should have gone
      int moved = 0, taken[W] = {0}, last = -1;
      for (int t = 0, from = 0; t < W; ++t) {
        if (t < from || !wants[w.r][t][taken[t]]) continue;
        moved |= 1 << t;
        last = t;
        from = t + 1;
        for (int i = t; i < W; ++i) ++taken[i];
      }
      if (scores) { if (last >= 0 && w.known != version(w.r, last, 0)) ++fails; }
      else {
        const int b = kNewsMovedBit;
        if (news_of_round(w.said[0] >> b, w.said[1] >> b, w.said[2] >> b, w.said[3] >> b) != moved) ++fails;
        for (int i = 0; i < W; ++i) {
          if (w.seen[i] != version(w.r, i, taken[i])) ++fails;
          if ((moved >> i & 1) && factors[w.r & 1][i] != version(w.r, i, 0)) ++fails;
        }
      }
      w.at = 0;
      if (++w.r == kRounds) w.done = true;
      break;
    }
  }
}

// late: the wave that only runs when no other can (kWaves: whichever the dice say); keen: one that runs whenever it can
static void run(int late, int keen) {
  for (int i = 0; i < kWaves; ++i) { waves[i] = Wave(); waves[i].id = i; }
  for (;;) {
    int ready[kWaves], n = 0, waiting = 0, done = 0;
    for (int i = 0; i < kWaves; ++i) {
      if (waves[i].done) ++done;
      else if (waves[i].waits) ++waiting;
      else ready[n++] = i;
    }
    if (done == kWaves) return;
    if (n == 0) {
      if (done || waiting < kWaves) { ++fails; return; }   // the others never come
      for (int i = 0; i < kWaves; ++i) {
        if (waves[i].label != waves[0].label) { ++fails; return; }
        waves[i].waits = false;
      }
      continue;
    }
    int pick = ready[draw(n)];
    for (int i = 0; i < n; ++i) if (ready[i] == keen) pick = keen;
    if (pick == late && n > 1) pick = ready[pick == ready[0] ? 1 : 0];
    step(waves[pick]);
  }
}

int main() {
  for (int seed = 1; seed <= 4000; ++seed)
    for (int late = 0; late <= kWaves; ++late) {
      state = seed * 0x9e3779b97f4a7c15ull;
      const int often = 2 + draw(5);
      for (auto& round : wants) for (auto& tile : round) for (bool& x : tile) x = draw(often) == 0;
      run(late, draw(kWaves + 1));
    }
  printf("%d failures\n", fails);
  return fails != 0;
}
"""


def test_all_waves_go_through_a_round_alike(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "news.cpp", tmp_path / "news"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-O1", "-std=c++17", "-I", os.path.join(ROOT, "ringattention_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout
