// gdem_chunks.h -- how the host cuts the steps of a packed gdem_step call into
// chunks (a rebuild offered, then steps).  No HIP: the policy is host
// arithmetic on what the device reports.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace gdem {

// Most steps of a chunk, and steps of a group (chunks launched together).
constexpr int kChunkSteps = 16;
// Steps launched on one estimate before the progress is read, and the gap a
// read leaves, in us.
constexpr int kReadSteps = 1024;
constexpr double kReadUs = 40.;

// Chooses the length of the chunks and the number of groups to launch.  A
// chunk in which a rebuild falls due leaves its remaining steps undone, each
// at the price of its empty launches, and every chunk pays the rebuild kernels
// that exit: long lives of the lists take long chunks, short lives short ones.
struct ChunkPolicy {
  double steps = 0., rebuilds = 0.;   // of the last few rebuilds
  double done = 0., launched = 0.;    // steps of the last groups at this length
  int32_t length = kChunkSteps;

  // Steps per rebuild; 0: not known yet.
  double life() const { return rebuilds >= 2. ? steps / rebuilds : 0.; }

  // The rebuild kernels of a chunk that exit, and an empty step, in us; one: a
  // step is one kernel.  Steps of a gas in chunks of 16, 8, 4, 2 and 1, us:
  // 100,000 spheres, 12 steps per rebuild 27.4, 27.8, 29.4, 31.4, 35.9; 4.5
  // steps 38.7, 35.7, 37.1, 39.3, 43.4; 1.1 steps 83, 73, 68, 67, 69.  1M: 40
  // steps 106.5, 107.2, 108.7, 110.9, 116.8; 1 step 534, 495, 474, 463, 457.
  static double offer_us(bool one) { return one ? 8.5 : 10.; }
  static double empty_us(bool one) { return one ? 1.2 : 4.; }

  // Cost of the launches a life takes beside its steps' work in chunks of c:
  // m chunks, of which the last ends wherever the rebuild falls.
  static double cost(int c, double life, bool one) {
    const double m = std::max(1., life / c + 0.5 * (1. - 1. / c));
    return offer_us(one) * m + empty_us(one) * std::max(0., m * c - life);
  }

  // Length of the next chunks (a power of two); one: a step is one kernel.
  int32_t choose(bool one) {
    int32_t best = kChunkSteps;
    const double l = std::max(life(), 1.);
    if (rebuilds >= 2.)
      for (int32_t c = kChunkSteps / 2; c >= 1; c /= 2)
        if (cost(c, l, one) < cost(best, l, one)) best = c;
    if (best != length || launched == 0.) {
      length = best;
      launched = kChunkSteps;
      done = rebuilds >= 2. ? launched * l / (l + 0.5 * (length - 1)) : launched;
    }
    return length;
  }

  // Length of the chunks of the last `left` < kChunkSteps steps: each rebuild
  // inside a chunk costs a read and further launches, chunks of one step none.
  int32_t tail(int32_t left, bool one) const {
    int32_t best = kChunkSteps;
    if (rebuilds < 2.) return best;
    const double due = left / std::max(life(), 1.);
    auto at = [&](int c) {
      return offer_us(one) * ((left + c - 1) / c) + due * (1. - 1. / c) * kReadUs;
    };
    for (int32_t c = kChunkSteps / 2; c >= 1; c /= 2)
      if (at(c) < at(best)) best = c;
    return best;
  }

  // Groups of kChunkSteps launched steps for `left` >= kChunkSteps steps: those
  // the last yield asks for, but never many more than the steps that are left,
  // and never more than kReadSteps.  The last one is left out where it is hardly
  // needed, or where what it would launch for nothing costs more than reading
  // the progress once more.
  int32_t groups(int32_t left, bool one) const {
    const double full = (double)left / kChunkSteps;
    const double want = std::min(full * launched / std::max(done, 1.), 1.3 * full + 1.);
    int32_t g = (int32_t)want;
    const double rest = want - g, over = (1. - rest) * kChunkSteps;
    if (rest > 0.1 && over * (offer_us(one) / length + empty_us(one)) < kReadUs) ++g;
    return std::max(1, std::min(g, kReadSteps / kChunkSteps));
  }

  // What the launches since the last call did: steps, steps launched by the
  // chunks that found any left to do (0: not whole groups), rebuilds.
  void note(int32_t did, int32_t offered, int32_t built) {
    if (offered > 0) {
      if (launched > 512.) {
        launched *= 0.5;
        done *= 0.5;
      }
      launched += offered;
      done += did;
    }
    if (built >= 4) {  // enough to judge by alone
      steps = did;
      rebuilds = built;
      return;
    }
    if (rebuilds > 8.) {
      steps *= 0.5;
      rebuilds *= 0.5;
    }
    rebuilds += built;
    steps = std::min(steps + did, 256. * std::max(rebuilds, 1.));
  }
};

}  // namespace gdem
