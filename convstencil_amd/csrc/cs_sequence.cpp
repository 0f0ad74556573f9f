// cs_sequence.cpp -- which kernels run a number of steps of a 2-D or 3-D FP64 grid.
//
// Four families compete (radius-1 box and star, radius-3 star and box): MFMA tables (mf 4),
// register-streaming strips (mf 7), level-pipelined strips (mf 10) and register tiles (mf 11), each
// at several depths.  Which is the fastest depends on both sides of the grid (strips and tiles that
// overlap, chunks of few rows), on the number of steps (what is left over runs shallow) and on the
// halo, so no line by the number of cells separates them: with such lines 48 steps of a radius-3 star on
// 2333 x 1500 took 948 us in tiles against 473 in strips, a radius-1 star on 21153 x 520 363 in
// pipelines against 318, a single step of the radius-3 star on 300 x 517 13.0 against 6.4, three of its
// box on 4096^2 245 against 172.  Here every launch's time is predicted from what bounds its family and
// the sequence of the least sum is taken.
//
// The predictions are fitted to launches of every variant on 360 grids (zero halo) and 90 grids (uploaded
// halo) of 96 to 20000 rows and columns, up to 105 M cells, and to strips on 110 narrow ones, one
// variant at a time on a warm card; rms error 2-6% for the pipelines, 4-6% for the tiles, 3-7% for the
// tables, 4-6% for the strips on grids 900 or more columns wide and 10% on narrower ones.
#include "cs_sequence.h"

#include <algorithm>
#include <cmath>
#include <limits>

namespace cs {

namespace {

constexpr double kCus = 256.0;
constexpr double kInf = std::numeric_limits<double>::infinity();

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Level-pipelined strips: all workgroups are resident and last as long as one chunk's rows: a + c rows
// (us), and `far` for every 100 MB beyond 200 MB of the grid's reads and writes; or the bytes at `tbs`.
// `block` = rows between barriers, `per_cu` = workgroups per CU.
struct PipeFit {
  int id, block, per_cu;
  double a, c, far, tbs, halo_a, halo_c;
};
const PipeFit kPipe[] = {
    {901004, 2, 2, 1.7, 0.660, 5.8, 4.46, 3.3, 0.784},  {901008, 2, 2, 0.0, 0.950, 2.1, 4.2, 2.0, 1.12},
    {901012, 2, 2, 1.6, 1.21, 2.6, 4.2, 4.0, 1.43},     {911004, 2, 2, 1.0, 0.616, 7.2, 4.91, 4.2, 0.693},
    {911008, 2, 2, 1.6, 0.676, 4.9, 4.49, 3.1, 0.919},  {911012, 2, 2, 0.6, 0.838, 2.6, 4.03, 4.5, 1.11},
    {911016, 2, 2, 0.0, 1.01, 3.7, 4.2, 4.1, 1.36},     {903002, 1, 2, 30.0, 0.997, 5.4, 7.58, 28.4, 1.20},
    {903004, 1, 2, 5.6, 1.87, 3.8, 4.2, 2.3, 2.16},     {913004, 2, 2, 4.0, 0.860, 6.0, 4.23, 0.0, 0.983},
    {913008, 2, 1, 2.5, 0.683, 4.1, 4.2, 0.5, 0.828},
};

double pipe_us(const Variant &v, const PipeFit &f, int64_t ny, int64_t nx, bool zero) {
  const int64_t strips = 1 + ceil_div(nx - 64 * v.px, v.bx), h = v.R * v.kf;
  const int64_t chunks = std::max<int64_t>(1, std::min<int64_t>(ny, (int64_t)kCus * f.per_cu / strips));
  const int64_t period = reg_period(v.R, v.st);
  const int64_t rows = ceil_div(ceil_div(ny, chunks) + 2 * h + (v.nw - 1) * f.block + 1, period) * period;
  const double mb = 16e-6 * (double)ny * (double)nx;
  const double t = zero ? f.a + f.c * (double)rows + f.far * std::max(0.0, mb - 200.0) / 100.0
                        : f.halo_a + f.halo_c * (double)rows;
  return std::max(t, mb / f.tbs);
}

// Register tiles: a launch, the tiles' bytes, the edge tiles' look at the halo and, with m tiles on a CU, a
// start for each of them and kf steps of a chain and m tiles' issue.
struct TileFit {
  int R, shape, rows;
  double a, each, mb, edge, lat, issue;
};
const TileFit kTile[2][5] = {
    {{1, SHAPE_BOX, 4, 4.45, 0.0, 0.108, 0.549, 0.229, 0.260},
     {1, SHAPE_BOX, 8, 5.14, 0.0, 0.113, 0.888, 0.297, 0.469},
     {1, SHAPE_STAR, 4, 4.31, 0.0, 0.118, 0.583, 0.257, 0.135},
     {1, SHAPE_STAR, 8, 4.60, 0.513, 0.113, 0.886, 0.344, 0.221},
     {3, SHAPE_STAR, 8, 4.81, 5.0, 0.107, 3.70, 0.210, 1.98}},
    {{1, SHAPE_BOX, 4, 5.67, 0.0, 0.105, 1.61, 0.365, 0.331},
     {1, SHAPE_BOX, 8, 6.88, 0.0, 0.118, 2.72, 0.661, 0.613},
     {1, SHAPE_STAR, 4, 5.17, 0.0, 0.112, 1.41, 0.328, 0.194},
     {1, SHAPE_STAR, 8, 6.34, 0.0, 0.130, 2.51, 0.701, 0.346},
     {3, SHAPE_STAR, 8, 8.0, 5.0, 0.101, 7.51, 0.496, 2.56}},
};

double tile_us(const Variant &v, const TileFit &f, int64_t tiles, int64_t edge, double cells) {
  const double cu = (double)ceil_div(tiles, (int64_t)kCus), mb = 8e-6 * ((double)tiles * v.by * v.bx + cells);
  return f.a + f.each * cu + f.mb * mb + f.edge * (double)edge / kCus + v.kf * (f.lat + f.issue * cu);
}

double tile_us(const Variant &v, const TileFit &f, int64_t ny, int64_t nx) {
  const int64_t tx = 1 + ceil_div(nx - v.bx, v.bx - 2 * v.R * v.kf), ty = 1 + ceil_div(ny - v.by, v.by - 2 * v.R * v.kf);
  double t = tile_us(v, f, tx * ty, std::min<int64_t>(tx, 2) * ty, (double)ny * (double)nx);
  // one or two steps with several tiles on a CU, and on narrow grids, where every tile looks at the halo:
  // 7219 x 135, 2 steps, 14.0 us against 11.0 in strips
  if (v.kf < 3 && tx <= 2 && ty > 16)
    t += 6.0;
  else if (v.kf < 3 && tx * ty > (int64_t)kCus)
    t += 4.0;
  return t;
}

const TileFit *tile_fit(const Variant &v, bool zero) {
  for (const TileFit &f : kTile[zero ? 0 : 1])
    if (f.R == v.R && f.shape == v.shape && f.rows == v.st) return &f;
  return nullptr;
}

// Register-streaming strips (zero halos): the longest edge or inner chunk or the sum of all rows over 1024
// SIMDs, and the bytes beyond what the caches hold, slower by the share of edge strips, whose rows are
// loaded cell by cell; the two overlap in part (norm q).
struct StripFit {
  int id, waves;  // waves per SIMD
  double a, edge, inner, edge_sum, inner_sum, tbs, mb, q, edge_bytes;
};
const StripFit kStrip[] = {
    {700402, 2, 6.0, 0.156, 0.368, 0.435, 0.550, 3.84, 78.6, 20, 0.438},
    {700404, 2, 4.9, 0.672, 0.699, 0.552, 0.475, 3.88, 65.5, 20, 0.537},
    {780408, 2, 15.0, 0.957, 1.16, 0.934, 0.748, 7.00, 206, 1.87, 1.14},
    {760208, 3, 9.5, 0.503, 0.477, 0.331, 0.231, 6.54, 179, 1.2, 0.589},
    {710402, 2, 5.4, 0.173, 0.400, 0.429, 0.555, 3.85, 77.1, 20, 0.422},
    {710404, 2, 7.7, 0.229, 0.618, 0.397, 0.423, 3.83, 79.7, 10.8, 0.508},
    {713202, 4, 15.0, 0.452, 0.985, 0.394, 0.256, 3.52, 68.9, 20, 1.60},
    {713203, 3, 15.0, 0.329, 0.623, 0.312, 0.188, 3.97, 49.2, 20, 0.664},
    {713204, 2, 15.0, 0.440, 0.460, 0.364, 0.263, 7.00, 143, 1.31, 0.613},
    {713206, 2, 15.0, 0.872, 0.041, 0.654, 0.462, 7.00, 245, 1.47, 1.08},
};

double strip_us(const Variant &v, const StripFit &f, int64_t ny, int64_t nx) {
  const int64_t period = reg_period(v.R, v.st), warm = 2 * v.R * v.kf;
  const RegSplit sp = reg_split(ny, nx, v.bx, v.R * v.kf, 1024 * f.waves, reg_edge_cost(v.px, v.R),
                                reg_least(v.R, v.kf, v.st));
  const int64_t ne = sp.strips >= 2 ? 2 : 1, ni = sp.strips - ne;
  const int64_t er = ceil_div(std::min(sp.he, ny) + warm, period) * period;
  const int64_t ir = sp.hm > 0 && ni > 0 ? ceil_div(std::min(sp.hm, ny) + warm, period) * period : 0;
  const double es = (double)((ne * sp.we + ni * (sp.hm > 0 ? 2 : sp.wi)) * er) / 1024.0;
  const double is = (double)((sp.hm > 0 ? ni * std::max<int64_t>(0, sp.wi - 2) : 0) * ir) / 1024.0;
  const double chain = std::max(f.edge * (double)er, f.inner * (double)ir);
  const double bytes = std::max(0.0, 16e-6 * (double)ny * (double)nx - f.mb) / f.tbs *
                       (1.0 + f.edge_bytes * std::min(1.0, 2.0 / (double)sp.strips));
  const double rows = std::max(chain, f.edge_sum * es + f.inner_sum * is);
  return f.a + std::pow(std::pow(rows, f.q) + std::pow(bytes, f.q), 1.0 / f.q);
}

// MFMA tables: tiles per CU, partly as whole rounds, or bytes; the single steps read either halo.
struct MfmaFit {
  int id;
  double a, tile, smooth, tbs, mb;
};
const MfmaFit kMfma[] = {
    {711101, 3.46, 2.44, 0.15, 4.27, 56.2}, {711111, 3.36, 2.32, 0.195, 4.31, 60.7}, {713101, 3.42, 4.80, 0.083, 3.94, 60.0},
    {13102, 4.75, 7.08, 0.0, 3.74, 59.8},   {13103, 5.81, 10.5, 0.017, 2.05, 30.5},  {713111, 3.94, 2.76, 0.0, 4.07, 43.9},
};

double mfma_us(const Variant &v, const MfmaFit &f, int64_t ny, int64_t nx) {
  const double n = (double)(ceil_div(ny, v.by) * ceil_div(nx, v.bx)) / kCus;
  const double t = f.a + f.tile * (f.smooth * std::max(1.0, n) + (1.0 - f.smooth) * std::ceil(n));
  return std::max(t, (16e-6 * (double)ny * (double)nx - f.mb) / f.tbs);
}

template <class T, size_t N>
const T *by_id(const T (&t)[N], int id) {
  for (const T &f : t)
    if (f.id == id) return &f;
  return nullptr;
}

}  // namespace

double launch_us_2d(const Variant &v, int64_t ny, int64_t nx, bool zero) {
  if (v.mf == 10) {
    const PipeFit *f = by_id(kPipe, v.id);
    return f && nx >= 64 * v.px ? pipe_us(v, *f, ny, nx, zero) : kInf;
  }
  if (v.mf == 11) {
    // 12 M cells: the largest grid fitted; the pipelines are twice as fast there
    if (ny < v.by || nx < v.bx || (double)ny * (double)nx > 12e6) return kInf;
    const TileFit *f = tile_fit(v, zero);
    return f ? tile_us(v, *f, ny, nx) : kInf;
  }
  if (v.mf == 7) {
    const StripFit *f = by_id(kStrip, v.id);
    return f && zero ? strip_us(v, *f, ny, nx) : kInf;
  }
  if (v.mf == 4) {
    const MfmaFit *f = by_id(kMfma, v.id);
    return f && (zero || v.kf == 1) ? mfma_us(v, *f, ny, nx) : kInf;
  }
  return kInf;
}

double tiles_us_2d(const Variant &v, int64_t tiles, int64_t edge, double cells) {
  const TileFit *f = tile_fit(v, true);
  return f ? tile_us(v, *f, tiles, edge, cells) : kInf;
}

bool Sequence2D::init(int R, int shape, int64_t ny, int64_t nx, bool zero) {
  if (ny < 1 || nx < 1) return false;
  zero_ = zero;
  std::fill(depth_, depth_ + kDepths + 1, nullptr);
  std::fill(tile_, tile_ + kDepths + 2, nullptr);
  double least[kDepths + 1];
  std::fill(least, least + kDepths + 1, kInf);
  bool newer = false;  // a pipeline or a tile fits
  const Variant *(*const lists[])(int *) = {variants_2d_f64, variants_2d_reg,
                                            R == 1 ? variants_2d_pipe_r1 : variants_2d_pipe_r3, variants_2d_block};
  for (auto list : lists) {
    int n = 0;
    const Variant *vs = list(&n);
    for (int i = 0; i < n; ++i) {
      const Variant &v = vs[i];
      if (v.R != R || v.shape != shape || v.kf > kDepths) continue;
      const double us = launch_us_2d(v, ny, nx, zero);
      if (!(us < kInf)) continue;
      newer = newer || v.mf >= 10;
      if (v.mf == 4 && v.kf == 1) {
        one_ = &v;
        one_us_ = us;
        if (!zero) continue;  // not before another launch
      }
      if (us < least[v.kf]) {
        least[v.kf] = us;
        depth_[v.kf] = &v;
      }
    }
  }
  if (!newer || !one_) return false;
  bulk_ = one_;
  bulk_us_ = one_us_;
  for (int k = 1; k <= kDepths; ++k)
    if (least[k] / k < bulk_us_ / bulk_->kf) {
      bulk_us_ = least[k];
      bulk_ = depth_[k];
    }
  if (bulk_->mf == 11) {
    int n = 0;
    const Variant *vs = variants_2d_block(&n);
    for (int i = 0; i < n; ++i) {
      if (vs[i].prepare != bulk_->prepare) continue;  // one kernel serves a tile's depths
      tile_[vs[i].kf] = &vs[i];
      tile_us_[vs[i].kf] = launch_us_2d(vs[i], ny, nx, zero);
    }
  }
  for (int e = 0; e < 2; ++e)
    for (int s = 0; s <= kSteps; ++s) {
      us_[e][s] = s == 0 && e == 0 ? 0.0 : kInf;
      pick_[e][s] = 0;
    }
  for (int s = 1; s <= kSteps; ++s)
    for (int e = 0; e < (zero ? 1 : 2); ++e)
      for (int k = 1; k <= kDepths && k <= s; ++k) {
        if (!depth_[k]) continue;
        const double us = us_[zero || k % 2 ? e : e ^ 1][s - k] + least[k];
        if (us < us_[e][s]) {
          us_[e][s] = us;
          pick_[e][s] = (signed char)k;
        }
      }
  return true;
}

// As few different depths as the number of steps allows: one or two next to one another.
Sequence2D::Cut Sequence2D::even_cut(int64_t steps) const {
  Cut best{kInf, 0, 0, 0, 0};
  if (bulk_->mf != 11) return best;
  for (int ones = 0; ones < (zero_ ? 1 : 2) && ones < steps; ++ones) {
    const int64_t s = steps - ones, last = ceil_div(s, bulk_->kf) + 2;
    for (int64_t n = s > kSteps ? ceil_div(s, bulk_->kf + 1) : 1; n <= last && n <= s; ++n) {
      const int64_t d = s / n, deeper = s % n;
      if (d + (deeper > 0) > kDepths || !tile_[d] || (deeper > 0 && !tile_[d + 1])) continue;
      const int64_t even = d % 2 == 0 ? n - deeper : deeper;
      if (!zero_ && even % 2) continue;
      const double us = (double)(n - deeper) * tile_us_[d] + (deeper > 0 ? (double)deeper * tile_us_[d + 1] + kSwitchUs : 0.0) +
                        ones * (one_us_ + kSwitchUs);
      if (us < best.us) best = Cut{us, n, deeper, ones, (int)d};
    }
  }
  return best;
}

bool Sequence3D::init(int R, int shape, int64_t nz, int64_t ny, int64_t nx) {
  std::fill(depth_, depth_ + kDepths + 1, nullptr);
  std::fill(us_, us_ + kDepths + 1, kInf);
  bulk_ = nullptr;
  int n = 0;
  const Variant *vs = variants_3d_tile(&n);
  for (int i = 0; i < n; ++i) {
    const Variant &v = vs[i];
    if (v.R != R || v.shape != shape || v.kf < 2 || v.kf > kDepths || nz < 1 || nx < v.bx || ny < v.by) continue;
    const double us = tile3_cost(v, nz, ny, nx) * v.kf;
    if (us < us_[v.kf]) {
      us_[v.kf] = us;
      depth_[v.kf] = &v;
    }
  }
  for (int k = 2; k <= kDepths; ++k)
    if (depth_[k] && (!bulk_ || us_[k] / k < us_[bulk_->kf] / bulk_->kf)) bulk_ = depth_[k];
  // the other depths on the same tile unless another one is predicted to be 15% faster (star 10 x 2000 x 66, 5
  // steps, 36.3 us on one tile, 40.0 on two)
  for (int i = 0; bulk_ && i < n; ++i) {
    const Variant &v = vs[i];
    if (v.R != R || v.shape != shape || v.by != bulk_->by || v.nw != bulk_->nw || v.kf < 2 || v.kf > kDepths) continue;
    const double us = tile3_cost(v, nz, ny, nx) * v.kf;
    if (us <= 1.15 * us_[v.kf]) {
      us_[v.kf] = us;
      depth_[v.kf] = &v;
    }
  }
  return depth_[2] && depth_[3];  // together they make every number from 2 up
}

double Sequence3D::cost(const int64_t *count) const {
  double us = -4.0;  // every change of variant counts as in two dimensions (Sequence2D)
  for (int k = 2; k <= kDepths; ++k)
    if (count[k] > 0) us += (double)count[k] * us_[k] + 4.0;
  return us;
}

// As few launches as the main depth allows, cut evenly, unless another mix is predicted to be 5% faster.  An
// odd number of steps never leaves one for the single-step kernel: radius-1 star 30 x 24 x 1000, 3 steps as
// 2 + 1 72 us, as one launch 18.
void Sequence3D::choose(int64_t steps, int64_t *count) const {
  const int kf = bulk_->kf;
  double least = kInf;
  const int64_t launches = ceil_div(steps, kf), d = steps / launches, deeper = steps % launches;
  if (d >= 2) {
    count[d] = launches - deeper;
    if (deeper > 0) count[d + 1] = deeper;
    least = 0.95 * cost(count);
  }
  const int64_t n = steps > kSteps ? ceil_div(steps - kSteps, kf) : 0;
  const int rest = (int)(steps - n * kf);
  for (int four = 0; 4 * four <= rest && (four == 0 || depth_[4]); ++four)
    for (int three = 0; 4 * four + 3 * three <= rest; ++three) {
      const int left = rest - 4 * four - 3 * three;
      if (left % 2) continue;
      int64_t c[kDepths + 1] = {0, 0, left / 2, three, four};
      c[kf] += n;
      const double us = cost(c);
      if (us < least) {
        least = us;
        std::copy(c, c + kDepths + 1, count);
      }
    }
}

}  // namespace cs
