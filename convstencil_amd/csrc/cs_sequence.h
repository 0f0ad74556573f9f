// cs_sequence.h -- launch sequences of least predicted time for 2-D and 3-D FP64 grids (cs_sequence.cpp).
#pragma once
#include "cs_internal.h"

namespace cs {

// Predicted us of one launch of a 2-D FP64 kernel over ny x nx interior cells; `zero`: every halo cell is
// +0.  Infinite for a kernel without a prediction or one that the grid does not fit.
double launch_us_2d(const Variant &v, int64_t ny, int64_t nx, bool zero);

// The same for one launch of a register-tile kernel over the tiles of several grids with +0 halos: `edge` of them
// in the first or last tile column, `cells` in all grids together.
double tiles_us_2d(const Variant &v, int64_t tiles, int64_t edge, double cells);

// The launches of any number of steps on one grid, zero halo or not.  Nothing is allocated.
class Sequence2D {
 public:
  // False where the stencil has no level-pipelined or register-tile kernel or none fits the grid.
  bool init(int R, int shape, int64_t ny, int64_t nx, bool zero);

  // The variant of the least time per step, and the single-step kernel (the only one that reads its
  // input buffer's halo whatever the state's buffer: it ends the sequence).
  const Variant *main() const { return bulk_; }
  const Variant *one() const { return one_; }

  // f(variant, count) for consecutive launches, in order.
  template <class F>
  void each(int64_t steps, F f) const {
    const int kf = bulk_->kf;
    const Cut c = even_cut(steps);
    if (c.us < kNever) {
      const Mix m = mixed(steps);
      if (c.us <= m.us) {
        if (c.deeper > 0) f(tile_[c.depth + 1], c.deeper);
        if (c.n > c.deeper) f(tile_[c.depth], c.n - c.deeper);
        if (c.ones > 0) f(one_, c.ones);
        return;
      }
    }
    const Mix m = split(steps);
    if (m.n > 0 && bulk_ != one_) f(bulk_, m.n);
    walk(m.fused, [&](const Variant *v) { f(v, (int64_t)1); });
    const int64_t ones = steps - m.n * kf - m.fused + (bulk_ == one_ ? m.n : 0);
    if (ones > 0) f(one_, ones);
  }

  // f(variant) for a variant of every kernel that a number of steps can take (a tile's depths share one).
  template <class F>
  void each_variant(F f) const {
    bool used[kDepths + 1] = {};
    for (int e = 0; e < 2; ++e)
      for (int i = 1; i <= kSteps; ++i) used[(int)pick_[e][i]] = true;
    f(one_);
    f(bulk_);
    for (int k = 1; k <= kDepths; ++k)
      if (used[k] && depth_[k] != bulk_ && depth_[k] != tile_[k]) f(depth_[k]);
  }

 private:
  // Steps that are put together from all depths; of more, the first go to the variant of the least time
  // per step.
  static constexpr int kSteps = 64, kDepths = 16;
  static constexpr double kNever = 1e300;
  // A launch after one of another kernel or depth waits for its code and finds its input in other XCDs' L2:
  // radius-1 box on 100 x 9000, launches of 9 and 11 steps by turns 34.7 us, two of 10 30.8, of 9 29.1.
  static constexpr double kSwitchUs = 4.0;

  // n launches of bulk_, `fused` steps by walk(), single steps for the rest.
  struct Mix {
    double us;
    int64_t n;
    int fused;
  };
  // n launches of a tile's kernel, of depth + 1 (the first `deeper`) and depth, then single steps.
  struct Cut {
    double us;
    int64_t n, deeper, ones;
    int depth;
  };

  Mix split(int64_t steps) const {
    const int kf = bulk_->kf;
    Mix m{0.0, steps > kSteps ? (steps - kSteps + kf - 1) / kf : 0, 0};
    if (!zero_ && kf % 2 == 0 && m.n % 2) ++m.n;  // an even number of even launches, see us_
    const int rest = (int)(steps - m.n * kf);
    m.fused = rest;
    if (!zero_)
      for (int i = 0; i < rest; ++i)
        if (us_[0][i] + (rest - i) * one_us_ < us_[0][m.fused] + (rest - m.fused) * one_us_) m.fused = i;
    m.us = m.n * bulk_us_ + us_[0][m.fused] + (rest - m.fused) * one_us_;
    return m;
  }
  // The same, the changes of variant included in its time.
  Mix mixed(int64_t steps) const {
    Mix m = split(steps);
    const Variant *seen[kDepths + 2];
    int variants = 0;
    auto add = [&](const Variant *v) {
      for (int i = 0; i < variants; ++i)
        if (seen[i] == v) return;
      seen[variants++] = v;
    };
    if (m.n > 0) add(bulk_);
    walk(m.fused, add);
    if (m.n * bulk_->kf + m.fused < steps) add(one_);
    m.us += kSwitchUs * (variants - 1);
    return m;
  }
  template <class F>
  void walk(int s, F f) const {
    for (int even = 0; s > 0;) {
      const Variant *v = depth_[(int)pick_[even][s]];
      f(v);
      s -= v->kf;
      if (!zero_) even ^= v->kf % 2 == 0;
    }
  }
  Cut even_cut(int64_t steps) const;

  bool zero_ = true;
  const Variant *depth_[kDepths + 1] = {};     // the fastest variant of each depth
  const Variant *tile_[kDepths + 2] = {};      // the depths of bulk_'s kernel, if that is a tile
  double tile_us_[kDepths + 1];
  const Variant *bulk_ = nullptr, *one_ = nullptr;
  double bulk_us_ = 0.0, one_us_ = 0.0;
  // us_[e][s]: the least time of s steps by launches of depth_, e = parity of the number of launches of
  // even depth; pick_: the depth of one of them.  A zero halo needs no parity (e = 0).  With another,
  // every launch but the single steps' reads each step's halo from that step's own buffer of the
  // ping-pong, and the state has to end in the buffer that as many single steps would leave it in:
  // a launch of even depth puts it into the other one.
  double us_[2][kSteps + 1];
  signed char pick_[2][kSteps + 1];
};

// The same for the stacked-wave 3-D kernels (k3d_tile.hip; zero halo): depths 2, 3 and, where compiled, 4,
// each on the tile of its least predicted time.  One step has no launch of theirs.
class Sequence3D {
 public:
  // False where no tile fits the grid.
  bool init(int R, int shape, int64_t nz, int64_t ny, int64_t nx);
  const Variant *main() const { return bulk_; }
  // f(variant, count) for consecutive launches of steps >= 2 steps.
  template <class F>
  void each(int64_t steps, F f) const {
    int64_t count[kDepths + 1] = {};
    choose(steps, count);
    for (int k = kDepths; k >= 2; --k)
      if (count[k] > 0) f(depth_[k], count[k]);
  }
  template <class F>
  void each_variant(F f) const {
    for (int k = 2; k <= kDepths; ++k)
      if (depth_[k]) f(depth_[k]);
  }

 private:
  static constexpr int kSteps = 24, kDepths = 4;
  // Launches per depth, and their time with the changes of variant.
  void choose(int64_t steps, int64_t *count) const;
  double cost(const int64_t *count) const;
  const Variant *depth_[kDepths + 1] = {};
  double us_[kDepths + 1];
  const Variant *bulk_ = nullptr;
};

}  // namespace cs
