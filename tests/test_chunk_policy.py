"""Length and number of the chunks the packed step is launched in (ChunkPolicy,
pacific_amd/csrc/gdem_chunks.h), built for the host and run against a model of
the device: a chunk offers a rebuild, then steps until the next rebuild falls
due; what is left of it is launched for nothing.

For lives of the lists from one step to hundreds the launches that do no work
(rebuild kernels that exit, empty steps) and the reads of the progress stay
near the least any fixed length of chunk needs, and below one rebuild offer per
step; after a change of the
life the launches on the old estimate stay bounded."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "pacific_amd", "csrc")

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include "gdem_chunks.h"
using namespace gdem;

// The device: rebuilds every life steps, give or take a quarter.
struct Device {
  double life, due = 0.;
  unsigned seed = 7;
  double next() {
    seed = seed * 1664525u + 1013904223u;
    return life * (0.75 + 0.5 * (seed >> 8) / 16777216.);
  }
  long offers = 0, empty = 0, steps = 0, reads = 0;   // of all calls
  int done = 0, target = 0, chunks = 0, rebuilds = 0;  // of this call
  void chunk(int len) {
    if (done >= target) {
      ++offers;
      empty += len;
      return;
    }
    ++chunks;
    bool built = false;
    if (due < 1.) {
      ++rebuilds;
      built = true;
      due += next() < 1. ? 1. : next();
    }
    if (!built) ++offers;
    for (int j = 0; j < len; ++j) {
      if (done >= target || (due < 1. && j)) { ++empty; continue; }
      ++done;
      ++steps;
      due -= 1.;
    }
  }
};

// One call of n steps; fixed > 0: chunks of that length, as many as the steps
// left (nothing launched on a guess).  Returns the launched steps.
long call(Device& d, ChunkPolicy& p, int n, bool one, int fixed) {
  d.done = d.chunks = d.rebuilds = 0;
  d.target = n;
  int done = 0, chunks = 0, rebuilds = 0, rounds = 0;
  long launched = 0;
  while (done < n) {
    if (++rounds > 10000) { printf("no progress\n"); exit(1); }
    const int left = n - done;
    const bool whole = left >= kChunkSteps;
    const int len = fixed ? fixed : whole ? p.choose(one) : p.tail(left, one);
    if (len < 1 || len > kChunkSteps || (len & (len - 1))) { printf("bad length %d\n", len); exit(1); }
    if (whole) {
      const int g = fixed ? left / kChunkSteps : p.groups(left, one);
      if (g < 1 || g > kReadSteps / kChunkSteps) { printf("bad groups %d\n", g); exit(1); }
      for (int k = 0; k < g; ++k)
        for (int j = 0; j < kChunkSteps; j += len) { d.chunk(len); launched += len; }
    } else {
      for (int k = left; k > 0; k -= len) { d.chunk(k < len ? k : len); launched += k < len ? k : len; }
    }
    ++d.reads;
    if (!fixed) p.note(d.done - done, whole ? (d.chunks - chunks) * len : 0, d.rebuilds - rebuilds);
    done = d.done;
    chunks = d.chunks;
    rebuilds = d.rebuilds;
  }
  return launched;
}

// us per step of launches without work and of reading the progress
double idle(const Device& d, bool one) {
  return (ChunkPolicy::offer_us(one) * d.offers + ChunkPolicy::empty_us(one) * d.empty +
          kReadUs * d.reads) / d.steps;
}

int main() {
  const double lives[] = {1., 1.3, 1.8, 2.7, 4., 5.5, 7., 10., 16., 25., 43., 60., 150., 400.};
  for (int one = 0; one < 2; ++one)
    for (double life : lives)
      for (int n : {1, 5, 40, 96, 500}) {
        double best = 1e30;
        for (int len = 1; len <= kChunkSteps; len *= 2) {
          Device d{life};
          ChunkPolicy p;
          for (int k = 0; k < 4000 / n + 4; ++k) call(d, p, n, one, len);
          best = best < idle(d, one) ? best : idle(d, one);
        }
        Device d{life};
        ChunkPolicy p;
        for (int k = 0; k < 4000 / n + 4; ++k) call(d, p, n, one, 0);
        printf("steady %d %g %d %.3f %.3f\n", one, life, n, idle(d, one), best);
      }
  // a phase of short lives, then one of long lives, and the other way round
  for (int one = 0; one < 2; ++one)
    for (int way = 0; way < 2; ++way) {
      Device d{way ? 60. : 2.};
      ChunkPolicy p;
      for (int k = 0; k < 20; ++k) call(d, p, 300, one, 0);
      d.life = way ? 2. : 60.;
      const long first = call(d, p, 300, one, 0);
      for (int k = 0; k < 4; ++k) call(d, p, 300, one, 0);
      const Device before = d;
      for (int k = 0; k < 10; ++k) call(d, p, 300, one, 0);
      d.offers -= before.offers; d.empty -= before.empty; d.steps -= before.steps; d.reads -= before.reads;
      printf("change %d %d %ld %.3f\n", one, way, first, idle(d, one));
    }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_chunks_follow_the_life_of_the_lists(tmp_path):
    src, exe = tmp_path / "chunks.cpp", tmp_path / "chunks"
    src.write_text(DRIVER)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-I", CSRC, "-o", str(exe), str(src)])
    steady = {}
    for line in subprocess.check_output([str(exe)]).decode().splitlines():
        kind, *v = line.split()
        if kind == "steady":
            one, life, n, got, best = int(v[0]), float(v[1]), int(v[2]), float(v[3]), float(v[4])
            steady[one, life, n] = got
            # within a fifth, or a microsecond a step, of the best fixed length
            assert got <= 1.2 * best + 1.0, line
            # no worse than a rebuild offered before every step
            assert got <= 1.15 * ((8.5 if one else 10.0) + 40.0 / n), line
        else:
            one, way, first, got = int(v[0]), int(v[1]), int(v[2]), float(v[3])
            # long after short lives: few launched for nothing; short (2 steps)
            # after long ones: a chunk of 16 for each at most
            assert first <= 300 * (16 / 2 if way else 1.5), line
            assert got <= 1.3 * steady[one, 1.8 if way else 60.0, 500] + 1.0, line
