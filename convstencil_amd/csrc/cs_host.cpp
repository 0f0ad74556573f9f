// cs_host.cpp -- host runtime and C ABI of libconvstencil (see include/convstencil.h).
//
// The reference's host launchers (src/2d/gpu.cu:245-333 and siblings) each build
// the B matrices, allocate two device buffers, copy the input, run the time loop
// of single-launch steps and copy the result back.  Here that body is a plan:
// buffers and B fragments are built once, the time loop is a sequence of fused
// launches (optionally captured in a hipGraph), and the reference-named
// launchers at the bottom of this file are thin wrappers that keep the
// reference's layouts, weight layouts and stdout lines.
#include "../../include/convstencil.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <map>
#include <string>
#include <vector>

#include "cs_host_util.h"
#include "cs_internal.h"
#include "cs_rng.h"
#include "cs_sequence.h"

using cs::Geo;
using cs::Variant;

using namespace cs::host;

struct cs_plan {
  cs_layout L{};
  int ndim = 0, R = 0, shape = 0;
  std::vector<double> w;  // dense weights
  cs_options opt{};
  int device = 0;
  hipStream_t stream = nullptr;
  double *buf[2] = {nullptr, nullptr};
  double *bfrag = nullptr;  // B fragments for the selected MFMA shape (or dense weights)
  int64_t frag_off = 0;     // when the register kernels' dense weights come first: where the
                            // MFMA single-step kernel's B fragments start (doubles)
  int cur = 0;              // buffer holding the current state
  int64_t steps_done = 0;
  bool halo_uniform = true;  // both buffers carry the same halo -> fusion is exact
  const Variant *vmain = nullptr;
  std::vector<const Variant *> vrem;  // vrem[r] runs r fused steps (r < vmain->kf), may be null
  const Variant *vone = nullptr;      // single-step variant (the register families use the MFMA one)
  const Variant *vzero = nullptr;     // with a zero halo in place of vmain, and its vrem (strip_of)
  std::vector<const Variant *> vzrem;
  // 2-D FP64 plans that choose for themselves: the sequences for a zero halo [1] and another one [0]
  bool by_time = false;
  cs::Sequence2D seq[2];
  bool by_time3 = false;  // 3-D ones on the stacked-wave kernels (zero halos)
  cs::Sequence3D seq3;
  std::map<std::pair<int64_t, int>, hipGraphExec_t> graphs;
  int64_t launches = 0;
  int tuned = 0;  // 0 defaults or a forced variant, 1 cached autotuner choice, 2 timed now
  // FP16 range guard: a bound on |cell| of both buffers (halo included) and the weights'
  // sum of magnitudes, which bounds each step's growth
  double amax = 0.0, wabs = 0.0;
};

namespace {

Geo make_geo(const cs_layout &L, const Variant *v) {
  Geo g{};
  for (int d = 0; d < 3; ++d) {
    g.ext[d] = L.ext[d];
    g.org[d] = L.org[d];
    g.n[d] = L.n[d];
  }
  g.tiles[0] = 1;
  g.tiles[1] = (L.n[1] + v->by - 1) / v->by;
  g.tiles[2] = (L.n[2] + v->bx - 1) / v->bx;
  return g;
}

// Default fusion depth when the caller does not choose one (the autotuner's
// cache, when present, overrides this).
// FP64 MFMA families (measured, GStencil/s per physical step): 1d1r 2^20 kf16 878 (kf32
// 842); box2d1r 10240^2 kf6 925-990 (kf4 861); star2d3r 8192^2 kf3 494 (kf2 454); box3d1r
// 512^3 kf1 260-265 (kf2 219); star3d1r kf2 303 (kf1 272).  Split precision: kf4 (2-D
// radius 1), kf2 (2-D radius 2-3 and 3-D).  The register kernels that pick_main prefers
// for 1-D and 2-D radius 1 choose their own depths there.
int default_kf(int ndim, int R, int top, int shape, bool fp64) {
  if (ndim == 1) return std::min(top, 16);
  if (ndim == 3) return std::min(top, fp64 && shape == cs::SHAPE3_BOX ? 1 : 2);
  if (!fp64) return std::min(top, R == 1 ? 4 : 2);
  return std::min(top, R == 1 ? 6 : 3);
}

std::vector<Variant> joined(std::initializer_list<const Variant *(*)(int *)> lists) {
  std::vector<Variant> v;
  for (auto f : lists) {
    int n = 0;
    const Variant *x = f(&n);
    v.insert(v.end(), x, x + n);
  }
  return v;
}

const Variant *family(int ndim, int *cnt, int prec = CS_PREC_FP64) {
  *cnt = 0;
  if (prec != CS_PREC_FP64)
    return ndim == 2 ? cs::variants_2d_split(cnt) : ndim == 3 ? cs::variants_3d_split(cnt) : nullptr;
  if (ndim < 1 || ndim > 3) return nullptr;
  // the MFMA kernels, then the --breakdown ladder's FMA kernels
  static const std::vector<Variant> all[3] = {
      joined({cs::variants_1d_reg, cs::variants_1d_f64, cs::variants_1d_ablation}),
      joined({cs::variants_2d_f64, cs::variants_2d_reg, cs::variants_2d_pipe_r1, cs::variants_2d_pipe_r3,
              cs::variants_2d_block,
              cs::variants_2d_stream, cs::variants_2d_ablation}),
      joined({cs::variants_3d_reg, cs::variants_3d_tile, cs::variants_3d_f64, cs::variants_3d_fma, cs::variants_3d_ablation})};
  *cnt = (int)all[ndim - 1].size();
  return all[ndim - 1].data();
}

// First variant of the family with this (MFMA shape or precision, radius, shape class,
// fusion depth) and, if st >= 0, this Variant::st; or the variant with id prefer_id.
const Variant *find_variant(int ndim, int mf, int R, int shape, int kf, int prefer_id, int prec = CS_PREC_FP64,
                            int st = -1) {
  int cnt = 0;
  const Variant *vs = family(ndim, &cnt, prec);
  const Variant *best = nullptr;
  for (int i = 0; i < cnt; ++i) {
    const Variant &v = vs[i];
    if (prefer_id > 0 && v.id == prefer_id && v.R == R && v.shape == shape) return &v;
    if (v.mf == mf && v.R == R && v.shape == shape && v.kf == kf && (st < 0 || v.st == st) && !best) best = &v;
  }
  return best;
}

int max_kf(int ndim, int mf, int R, int shape, int prec = CS_PREC_FP64, int st = -1) {
  int cnt = 0, m = 0;
  const Variant *vs = family(ndim, &cnt, prec);
  for (int i = 0; i < cnt; ++i)
    if (vs[i].mf == mf && vs[i].R == R && vs[i].shape == shape && (st < 0 || vs[i].st == st))
      m = std::max(m, vs[i].kf);
  return m;
}

// The single-step variant of an FP64 plan whose main variant is v: v itself when it is a
// single-step one (a variant forced by id must be the one that runs), else its family's
// first single-step variant -- except that the register kernels' single steps (alternating
// halos, remainders of one step) run on the LDS-staged MFMA single-step kernel, which keeps
// more bytes in flight: measured (GStencil/s) box2d1r 10240^2 300 against 203, star2d3r
// 8192^2 286 against 253, box2d3r 204 against 133 (1024^2 117 against 15).
const Variant *single_step(int nd, int R, int shape, const Variant *v) {
  if (v->kf == 1) return v;
  // the fused 3-D register and tile kernels: the 8 x 8 block single-step kernel (512^3: 258-268
  // GStencil/s against 242 for the register single step)
  if ((v->mf == 9 || v->mf == 12) && nd == 3)
    if (const Variant *m = find_variant(nd, 8, R, shape, 1, 0, CS_PREC_FP64)) return m;
  if (v->mf == 10 || ((v->mf == 6 || v->mf == 7) && !(nd == 2 && R > 1 && shape == cs::SHAPE_BOX)))
    if (const Variant *m = find_variant(nd, 4, R, shape, 1, 0, CS_PREC_FP64)) return m;
  if (v->mf == 10) return find_variant(nd, 7, R, shape, 1, 0, CS_PREC_FP64);
  if (v->mf == 11) return find_variant(nd, 11, R, shape, 1, 0, CS_PREC_FP64, v->st);
  return find_variant(nd, v->mf, R, shape, 1, 0, CS_PREC_FP64);
}

// 2-D grids of at most this many interior cells take depth 4 from the radius-1 box register
// kernels: their launches run short of waves and depth 8's longer tail dominates (2048^2:
// 825 GStencil/s at depth 4 against 635 at depth 8; 3072^2: 1136 against 1183).
constexpr int64_t kRegSmallGrid = 2560LL * 2560LL;

// Whether a variant can run an interior of ny rows of nx columns (the level-pipelined kernels' strips
// and the tiles of the register-tile and the stacked 3-D kernels lie inside the interior).
bool fits(const Variant *v, int64_t ny, int64_t nx) {
  if (v->mf == 12) return nx >= v->bx && ny >= v->by;
  return (v->mf != 10 && v->mf != 11) || (nx >= 64 * v->px && (v->mf != 11 || ny >= v->by));
}

// The variant that runs r steps left over by a main variant v; null where there is none.  The
// level-pipelined kernels are compiled for a few depths only; the register-streaming kernels
// fill in, for the radius-3 box, where those spill, the dilated tables (3 steps of 4096^2 171 us, as
// 2 + 1 188).
const Variant *remainder_variant(int nd, int R, int shape, const Variant *v, int r, int prec, int st) {
  if (prec == CS_PREC_FP64 && v->mf == 12) {  // the same tile's shallower variants
    int cnt = 0;
    const Variant *vs = cs::variants_3d_tile(&cnt);
    for (int i = 0; i < cnt; ++i)
      if (vs[i].shape == shape && vs[i].by == v->by && vs[i].nw == v->nw && vs[i].kf == r) return &vs[i];
    return nullptr;
  }
  if (prec != CS_PREC_FP64 && v->st == 3)  // the bits of depth 2: even depths, with its anchors above it
    return r > 1 && r % 2 ? nullptr : find_variant(nd, v->mf, R, shape, r, 0, prec, r > 2 ? 3 : 2);
  const Variant *u = find_variant(nd, v->mf, R, shape, r, 0, prec, v->mf == 11 && prec == CS_PREC_FP64 ? v->st : st);
  if (!u && prec == CS_PREC_FP64 && v->mf == 10)
    u = find_variant(nd, R > 1 && shape == cs::SHAPE_BOX ? 4 : 7, R, shape, r, 0, prec);
  return u;
}

// The level-pipelined kernel of the depth that the caller asks for, the family's own, on a grid of a size
// where it is the faster one (plans without a wish: cs_sequence.cpp), or null.  Measured, us per step
// of 96-step runs, other / this family: box r1 2048^2 5.0 / 5.3, 3072^2 8.2 / 7.4; star r1 3072^2
// 5.4 / 5.3; star r3 3072^2 13.1 / 13.9, 4096^2 19.0 / 17.9; box r3 3072^2 33.5 / 39.6, 4096^2 56.5 / 52.9.
const Variant *pick_pipe(int R, int shape, int fusion_depth, int64_t ny, int64_t nx) {
  const bool box = shape == cs::SHAPE_BOX;
  const int depth = R == 1 ? (box ? 12 : 16) : box ? 4 : 8;
  const int64_t least = R == 1 ? (box ? 5000000 : 8000000) : 14000000;
  if (nx < 512 || ny * nx < least || fusion_depth != depth) return nullptr;
  return find_variant(2, 10, R, shape, depth, 0);
}

// With a zero halo the radius-1 box runs faster in register-streaming strips of the same depth where the
// pipeline's wide strips overlap or are few: measured, us of 48 steps, strips / pipeline, 20000 x 520 418 / 531,
// 100000 x 520 1562 / 2068, 30000 x 1030 988 / 1031, 3000^2 315 / 360, 5000 x 2000 356 / 385, 3500^2 409 / 431, but
// 2300^2 260 / 259, 3600 x 4400 495 / 454, 12000 x 1500 597 / 604 (17 steps 291 / 275), 8192^2 1728 / 1519.  Else null.
const Variant *strip_of(const Variant *v, int fusion_depth, int64_t ny, int64_t nx) {
  if (v->mf != 10 || v->R != 1 || v->shape != cs::SHAPE_BOX || fusion_depth != v->kf) return nullptr;
  const int64_t cells = ny * nx;
  return nx <= 1100 || (cells >= 6000000 && cells < 13000000) ? find_variant(2, 7, 1, cs::SHAPE_BOX, v->kf, 0) : nullptr;
}

// Its r steps left over: eight in the pipeline (5000 x 2000 59 us, in strips 80; 20000 x 520 92, 96).
const Variant *strip_remainder(const Variant *strip, int r) {
  return r == 8 ? find_variant(2, 10, 1, cs::SHAPE_BOX, 8, 0)
                : remainder_variant(2, 1, cs::SHAPE_BOX, strip, r, CS_PREC_FP64, -1);
}

// The main variant of a plan: a forced id, else the preferred family's default depth (ny x nx = the
// interior of one grid, 0 when no single grid decides).
const Variant *pick_main(int nd, int R, int shape, int prec, int fusion_depth, int tile_variant, int64_t ny = 0,
                         int64_t nx = 0) {
  const int64_t cells = nd == 2 ? ny * nx : 0;
  const int mf = prec != CS_PREC_FP64 ? prec : 4;
  const Variant *v = nullptr;
  if (tile_variant > 0) {
    // a forced variant of the stencil's shape class, or a box variant (it computes any
    // stencil of its radius: the taps outside the stencil get zero weights)
    v = find_variant(nd, 0, R, shape, 0, tile_variant, prec);
    if (!v) v = find_variant(nd, 0, R, cs::SHAPE_BOX, 0, tile_variant, prec);
    if (v && nd >= 2 && prec == CS_PREC_FP64 && !fits(v, ny, nx)) v = nullptr;
  } else if (prec == CS_PREC_FP64) {
    if (nd == 2) v = pick_pipe(R, shape, fusion_depth, ny, nx);
    if (v) return v;
    // 1-D: the register-resident kernels (mf 6) at their deepest compiled fusion, else the
    // 4 x 4 x 4 blocks; 2-D: the register-streaming kernels (mf 7), else the dilated 8 x 8
    // blocks; 3-D: the fused register-streaming kernels (mf 9, radius 1), else the 8 x 8
    // block family (mf 8) where it exists, else the register-blocked FMA kernels (mf 3,
    // radius 2-3), else the 4 x 16 strips.  The 2-D box radius-3 register kernels spill; the
    // dilated tables are faster there (8192^2, 64 steps: 304-308 GStencil/s at depth 2-3
    // against 184-195).
    const bool reg2d = !(nd == 2 && R > 1 && shape == cs::SHAPE_BOX);
    const int fams[4] = {nd == 3 ? 9 : nd == 1 ? 6 : reg2d ? 7 : mf, nd == 3 ? 8 : mf, nd == 3 ? 3 : mf, mf};
    // a requested depth that some family compiles exactly is honoured exactly; single
    // steps of the register families run on the MFMA single-step kernel, as a plan's
    // remainders do (see single_step)
    if (fusion_depth > 0)
      for (int fmf : fams) {
        if (fusion_depth == 1 && (fmf == 6 || fmf == 7 || fmf == 9)) continue;
        if (!v) v = find_variant(nd, fmf, R, shape, fusion_depth, 0, prec);
      }
    for (int fmf : fams) {
      if (v) break;
      const int top = max_kf(nd, fmf, R, shape, prec);
      if (top == 0) continue;
      // register kernels (measured at 10240^2 / 8192^2, 64 steps): 2-D radius 1 depth 8
      // (1980-2001 GStencil/s; depth 12 1890-1908), star2d3r depth 4 (1016-1018; 3: 797,
      // 6: 761); 1-D the deepest compiled
      // the 3-D register kernels fuse two steps for the box and three for the star (512^3:
      // box 433-451 GStencil/s at depth 2 and 3 alike, star 621 at depth 3 against 449-472);
      // their single steps are slower than the 8 x 8 blocks', which a plan takes instead
      if (fmf == 9 && top < 2) continue;
      int kf = fusion_depth > 0 ? std::min(fusion_depth, top)
               : fmf == 6       ? top
               : fmf == 7       ? std::min(top, R == 1 ? (shape == cs::SHAPE_BOX && cells > 0 &&
                                                          cells <= kRegSmallGrid ? 4 : 8)
                                                 : shape == cs::SHAPE_STAR ? 4 : 2)
               : fmf == 9       ? std::min(top, shape == cs::SHAPE3_STAR ? 3 : 2)
                                : default_kf(nd, R, top, shape, true);
      for (; kf >= 1 && !v; --kf) v = find_variant(nd, fmf, R, shape, kf, 0, prec);
      if (v) break;
    }
  }
  return v;
}

// Prepares every variant that a sequence may take.
template <class S>
cs_status prepare_sequence(const S &s) {
  hipError_t e = hipSuccess;
  s.each_variant([&](const Variant *v) {
    if (e == hipSuccess) e = v->prepare();
  });
  CS_HIP(e);
  return CS_OK;
}

cs_status select_variants(cs_plan *p) {
  const int nd = p->ndim;
  const int prec = p->opt.precision;
  if (nd < 1 || nd > 3) return CS_ERR_UNSUPPORTED;
  if (prec != CS_PREC_FP64 && (prec < CS_PREC_BF16X3 || prec > CS_PREC_FP16W3)) return CS_ERR_INVALID;
  if (prec != CS_PREC_FP64 && nd == 1) return CS_ERR_UNSUPPORTED;
  // Split precision (Variant::mf holds the precision): the dilated form (st 2) for the
  // stencil's shape class, else its box variants (zero weights off the stencil), else the
  // Toeplitz form (st 0, box only).  The remainder launches come from the same form.
  const int mf = prec != CS_PREC_FP64 ? prec : 4;
  // The 49-point box in FP16 w3 and BF16x3 takes depth 6 with the anchors of depth 2 (st 3, see CfgS2):
  // below it a launch is bound by its bytes and its tile's load.  Measured, us a step at depth 2 and
  // 6 on 64 x 64 tiles and at depth 6 on 80 x 64: FP16 w3 300 x 517 5.14, 4.08, 4.52; 2048^2 16.7, 11.6,
  // 12.3; 4096^2 54.5, 39.9, 38.2; 8192^2 194.7, 131.9, 124.4; BF16x3 (64 x 64) 300 x 517 5.62, 4.58;
  // 8192^2 214.0, 166.6.
  const bool deep = nd == 2 && p->R == 3 && p->shape == cs::SHAPE_BOX && p->opt.fusion_depth == 0 &&
                    p->opt.tile_variant <= 0 && (prec == CS_PREC_FP16W3 || prec == CS_PREC_BF16X3);
  const Variant *v = nullptr;
  p->by_time = nd == 2 && prec == CS_PREC_FP64 && p->opt.fusion_depth == 0 && p->opt.tile_variant <= 0 &&
               p->seq[1].init(p->R, p->shape, p->L.n[1], p->L.n[2], true) &&
               p->seq[0].init(p->R, p->shape, p->L.n[1], p->L.n[2], false);
  // where a tile fits (64 columns, 24 rows) the other 3-D families lose on every grid measured, from 2% (box
  // 40 x 500 x 500) to 4.6 times (box 64^3 22 -> 4.9 us a step)
  p->by_time3 = nd == 3 && prec == CS_PREC_FP64 && p->opt.fusion_depth == 0 && p->opt.tile_variant <= 0 &&
                p->seq3.init(p->R, p->shape, p->L.n[0], p->L.n[1], p->L.n[2]);
  if (p->by_time) {
    v = p->seq[1].main();
  } else if (p->by_time3) {
    v = p->seq3.main();
  } else if (p->opt.tile_variant > 0) {
    v = pick_main(nd, p->R, p->shape, prec, p->opt.fusion_depth, p->opt.tile_variant, p->L.n[1], p->L.n[2]);
    if (!v) return CS_ERR_INVALID;
  } else if (prec == CS_PREC_FP64) {
    v = pick_main(nd, p->R, p->shape, prec, p->opt.fusion_depth, 0, p->L.n[1], p->L.n[2]);
  } else {
    const int tries[3][2] = {{p->shape, 2}, {cs::SHAPE_BOX, 2}, {cs::SHAPE_BOX, 0}};
    for (const auto &tr : tries) {
      const int top = max_kf(nd, mf, p->R, tr[0], prec, tr[1]);
      if (top == 0) continue;
      int kf = p->opt.fusion_depth > 0 ? std::min(p->opt.fusion_depth, top)
                                       : default_kf(nd, p->R, top, tr[0], false);
      if (deep && tr[0] == cs::SHAPE_BOX && tr[1] == 2)
        v = find_variant(nd, mf, 3, cs::SHAPE_BOX, 6,
                         prec == CS_PREC_FP16W3 && p->L.n[1] * p->L.n[2] >= 12000000 ? 3263406 : 0, prec, 3);
      for (; kf >= 1 && !v; --kf) v = find_variant(nd, mf, p->R, tr[0], kf, 0, prec, tr[1]);
      if (v) break;
    }
  }
  if (!v) return CS_ERR_UNSUPPORTED;
  p->shape = v->shape;
  const int fam = prec == CS_PREC_FP64 ? -1 : v->st == 3 ? 2 : v->st;
  p->vmain = v;
  // single-step launches: the chosen variant itself when it is a single-step one (a variant
  // forced by id must be the one that runs), else the family's first single-step variant
  p->vone = p->by_time              ? p->seq[1].one()
            : prec == CS_PREC_FP64 ? single_step(nd, p->R, p->shape, v)
            : v->kf == 1           ? v
                                   : find_variant(nd, v->mf, p->R, p->shape, 1, 0, prec, fam);
  if (!p->vone) return CS_ERR_UNSUPPORTED;
  p->vrem.assign(v->kf, nullptr);
  for (int r = 1; r < v->kf && !p->by_time && !p->by_time3; ++r)
    p->vrem[r] = remainder_variant(nd, p->R, p->shape, v, r, prec, fam);
  p->vzero = p->opt.tile_variant <= 0 && prec == CS_PREC_FP64 && nd == 2
                 ? strip_of(v, p->opt.fusion_depth, p->L.n[1], p->L.n[2])
                 : nullptr;
  p->vzrem.clear();
  for (int r = 0; p->vzero && r < v->kf; ++r)
    p->vzrem.push_back(r > 0 ? strip_remainder(p->vzero, r) : nullptr);
  for (const Variant *u : {p->vmain, p->vone, p->vzero})
    if (u) CS_HIP(u->prepare());
  for (const auto *rem : {&p->vrem, &p->vzrem})
    for (const Variant *u : *rem)
      if (u) CS_HIP(u->prepare());
  if (p->by_time) CS_TRY(prepare_sequence(p->seq[1]));
  if (p->by_time3) CS_TRY(prepare_sequence(p->seq3));
  if (prec != CS_PREC_FP64) {
    std::vector<unsigned char> hb(1 << 20);
    const size_t bytes = nd == 3      ? cs::build_bfrag_split3(prec, p->R, p->shape, p->w.data(), hb.data(), hb.size())
                         : v->st >= 2 ? cs::build_bfrag_split2(prec, p->R, p->shape, p->w.data(), hb.data(), hb.size())
                                      : cs::build_bfrag_split(prec, p->R, p->w.data(), hb.data(), hb.size());
    if (bytes == 0) return CS_ERR_UNSUPPORTED;
    if (p->bfrag) (void)hipFree(p->bfrag);
    p->bfrag = nullptr;
    CS_HIP(hipMalloc(&p->bfrag, bytes));
    CS_HIP(hipMemcpy(p->bfrag, hb.data(), bytes, hipMemcpyHostToDevice));
    return CS_OK;
  }
  // the FMA kernels (the ladder's, the 3-D mf 3 family, the register-streaming mf 7 and mf 9
  // families, the level-pipelined mf 10 family and the tiles of mf 11 and 12) read the dense weights (zero-padded to whole 64-entry rows); a plan of
  // those whose single steps run on an MFMA kernel (mf 7 and 10: the 2-D 4 x 4 x 4 kernel, mf 9
  // and 12: the 3-D 8 x 8 blocks) appends that kernel's B fragments
  p->frag_off = 0;
  if (p->by_time || v->mf == 1 || v->mf == 2 || v->mf == 3 || v->mf == 7 || v->mf == 9 || v->mf == 10 ||
      v->mf == 11 || v->mf == 12) {
    std::vector<double> h((p->w.size() + 63) / 64 * 64, 0.0);
    std::copy(p->w.begin(), p->w.end(), h.begin());
    if ((p->by_time || v->mf == 7 || v->mf == 10 || v->mf == 11) && p->vone->mf == 4) {
      p->frag_off = (int64_t)h.size();
      h.resize(h.size() + (size_t)cs::bfrag_ksteps_2d_f64(4, p->R, p->shape) * 64);
      cs::build_bfrag_2d_f64(4, p->R, p->shape, p->w.data(), h.data() + p->frag_off);
    } else if ((v->mf == 9 || v->mf == 12) && p->vone->mf == 8) {
      p->frag_off = (int64_t)h.size();
      h.resize(h.size() + (size_t)cs::bfrag_ksteps_3d2_f64(p->R, p->shape) * 64);
      cs::build_bfrag_3d2_f64(p->R, p->shape, p->w.data(), h.data() + p->frag_off);
    }
    if (p->bfrag) (void)hipFree(p->bfrag);
    p->bfrag = nullptr;
    CS_HIP(hipMalloc(&p->bfrag, h.size() * sizeof(double)));
    CS_HIP(hipMemcpy(p->bfrag, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
    return CS_OK;
  }
  // B fragments for the family's MFMA shape
  const int nks = nd == 1   ? cs::bfrag_ksteps_1d_f64(p->R)
                  : nd == 2 ? cs::bfrag_ksteps_2d_f64(v->mf, p->R, p->shape)
                  : v->mf == 8 ? cs::bfrag_ksteps_3d2_f64(p->R, p->shape)
                               : cs::bfrag_ksteps_3d_f64(p->R, p->shape);
  std::vector<double> h((size_t)nks * 64);
  if (nd == 1)
    cs::build_bfrag_1d_f64(p->R, p->w.data(), h.data());
  else if (nd == 2)
    cs::build_bfrag_2d_f64(v->mf, p->R, p->shape, p->w.data(), h.data());
  else if (v->mf == 8)
    cs::build_bfrag_3d2_f64(p->R, p->shape, p->w.data(), h.data());
  else
    cs::build_bfrag_3d_f64(p->R, p->shape, p->w.data(), h.data());
  if (p->bfrag) (void)hipFree(p->bfrag);
  p->bfrag = nullptr;
  CS_HIP(hipMalloc(&p->bfrag, h.size() * sizeof(double)));
  CS_HIP(hipMemcpy(p->bfrag, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
  return CS_OK;
}

// One launch of v; `done` = physical steps of the state's ping-pong so far.
cs_status launch_one(cs_plan *p, const Variant *v, int64_t done) {
  Geo g = make_geo(p->L, v);
  // step `done` reads the halo of buffer done & 1; with halos that differ, the level-pipelined
  // kernels are told when that is not the buffer that holds the state
  g.flip = p->halo_uniform ? 0 : (p->cur ^ done) & 1;
  const double *wts = (v->mf == 4 || v->mf == 8) && p->frag_off > 0 ? p->bfrag + p->frag_off : p->bfrag;
  CS_HIP(v->launch(p->buf[p->cur], p->buf[p->cur ^ 1], wts, g, p->stream));
  p->cur ^= 1;
  p->launches += 1;
  return CS_OK;
}

const Variant *main_variant(const cs_plan *p) { return p->halo_uniform && p->vzero ? p->vzero : p->vmain; }

// Whether the plan's launches may fuse steps: with halos that differ between the buffers only
// the level-pipelined and the register-tile kernels can (they read every level's halo from its
// own buffer).
bool fuses(const cs_plan *p) {
  return p->halo_uniform || (p->opt.precision == CS_PREC_FP64 && (p->vmain->mf == 10 || p->vmain->mf == 11));
}

// Steps per launch of a run of `steps` steps, as reported: the deepest launch's.
int32_t executed_depth(const cs_plan *p, int64_t steps) {
  if ((!p->by_time && !(p->by_time3 && p->halo_uniform)) || steps <= 0) return fuses(p) ? p->vmain->kf : 1;
  int d = 1;
  auto deepest = [&](const Variant *v, int64_t) { d = std::max(d, v->kf); };
  if (p->by_time)
    p->seq[p->halo_uniform].each(steps, deepest);
  else if (steps > 1)
    p->seq3.each(steps, deepest);
  return d;
}

// Launch sequence for `steps` physical steps.  With uniform halos, fused
// launches are exact: take the main depth as often as it fits, then the largest
// compiled depth that fits the rest.  Otherwise every launch is a single step so
// that each step reads the halo of its own buffer, as the reference's ping-pong
// does -- or, where the main variant is a level-pipelined kernel, launches of that family
// (all of even depth) and single steps for the rest.  After those the state must lie in
// the buffer whose halo it has by then, as after single steps: each even launch moves it to the
// other one, so their number has to be even.  Of an odd number the last that two smaller
// ones can replace is split, and if none can be, the last becomes single steps.  The single
// steps come last, when the state is back in its own buffer.
void plan_sequence(const cs_plan *p, int64_t steps, std::vector<const Variant *> *seq) {
  seq->clear();
  if (steps <= 0) return;
  if (p->by_time) {
    p->seq[p->halo_uniform].each(
        steps, [&](const Variant *v, int64_t n) { seq->insert(seq->end(), (size_t)n, v); });
    return;
  }
  if (p->by_time3 && p->halo_uniform && steps > 1) {
    p->seq3.each(steps, [&](const Variant *v, int64_t n) { seq->insert(seq->end(), (size_t)n, v); });
    return;
  }
  const Variant *vmain = main_variant(p);
  const std::vector<const Variant *> &vrem = vmain == p->vmain ? p->vrem : p->vzrem;
  if (!fuses(p) || vmain->kf == 1) {
    seq->assign((size_t)steps, p->vone);
    return;
  }
  const int kf = vmain->kf;
  if (p->opt.precision == CS_PREC_FP64 && (vmain->mf == 11 || vmain->mf == 12)) {
    // every depth is compiled (mf 12: from 2 up): as few launches as the main depth allows, cut
    // evenly.  With halos that differ an odd number of even depths k has one of them cut into k - 1
    // and 1.
    const int64_t n = (steps + kf - 1) / kf;
    int64_t even = 0;
    for (int64_t i = 0; i < n; ++i) {
      const int64_t d = steps / n + (i < steps % n);
      const Variant *u = d == kf ? vmain : vrem[(size_t)d];
      seq->push_back(u ? u : p->vone);
      even += d % 2 == 0;
    }
    if (!p->halo_uniform && even % 2) {
      size_t i = 0;
      while ((*seq)[i]->kf % 2) ++i;
      (*seq)[i] = vrem[(size_t)(*seq)[i]->kf - 1];
      seq->push_back(p->vone);
    }
    return;
  }
  seq->assign((size_t)(steps / kf), vmain);
  int64_t rem = steps % kf;
  while (rem > 0) {
    const Variant *best = p->vone;
    for (const Variant *u : vrem)
      if (u && u->kf <= rem && u->kf > best->kf && (p->halo_uniform || u->mf == 10)) best = u;
    seq->push_back(best);
    rem -= best->kf;
  }
  if (p->opt.precision == CS_PREC_FP64 && vmain->mf == 10 && steps > kf && steps % kf) {
    // a shallow last launch moves as many bytes as a deep one: kf + r steps are better cut
    // evenly (box r1 10240^2, 12 + 4 against 8 + 8 steps: 0.91 against 0.84 ms)
    const int r = (int)(steps % kf);
    for (int b = (kf + r) / 2; b > r; --b) {
      const Variant *u = kf + r - b < kf ? vrem[(size_t)(kf + r - b)] : nullptr, *v = vrem[(size_t)b];
      if (!u || !v || u->mf == 4 || (!p->halo_uniform && (u->mf != 10 || v->mf != 10))) continue;
      seq->resize((size_t)(steps / kf) - 1);
      seq->push_back(u);
      seq->push_back(v);
      break;
    }
  }
  if (p->halo_uniform) return;
  size_t n = 0;  // launches of the family come first
  while (n < seq->size() && (*seq)[n]->mf == 10) ++n;
  if (n % 2 == 0) return;
  for (size_t i = n; i-- > 0;) {
    const int k = (*seq)[i]->kf;
    for (int half = k / 2; half >= 1; --half) {
      const Variant *u = vrem[(size_t)half], *v = vrem[(size_t)(k - half)];
      if (!u || !v || u->mf != 10 || v->mf != 10) continue;
      (*seq)[i] = v;
      seq->insert(seq->begin() + (ptrdiff_t)n, u);
      return;
    }
  }
  const int k = (*seq)[n - 1]->kf;
  seq->erase(seq->begin() + (ptrdiff_t)(n - 1));
  seq->insert(seq->end(), (size_t)k, p->vone);
}

cs_status issue_steps(cs_plan *p, int64_t steps) {
  std::vector<const Variant *> seq;
  plan_sequence(p, steps, &seq);
  int64_t done = p->steps_done;
  for (const Variant *v : seq) {
    CS_TRY(launch_one(p, v, done));
    done += v->kf;
  }
  return CS_OK;
}

// Number of launches issue_steps() makes for `steps` steps.
int64_t count_launches(const cs_plan *p, int64_t steps) {
  std::vector<const Variant *> seq;
  plan_sequence(p, steps, &seq);
  return (int64_t)seq.size();
}

cs_status run_steps(cs_plan *p, int64_t steps) {
  if (steps < 0) return CS_ERR_INVALID;
  if (steps == 0) return CS_OK;
  double bound = 0.0;
  if (!fp16_range_ok(p->opt.precision, p->amax, p->wabs, steps, &bound)) {
    fprintf(stderr,
            "convstencil: FP16 split precision needs |values| < 2^15; the state may reach %.3g within %lld "
            "step(s)\n",
            bound, (long long)steps);
    return CS_ERR_INVALID;
  }
  p->amax = bound;
  if (p->L.n[0] == 0 || p->L.n[1] == 0 || p->L.n[2] == 0) {
    // no interior cell: every step only swaps the two buffers (no kernel has work)
    if (steps & 1) p->cur ^= 1;
    p->steps_done += steps;
    return CS_OK;
  }
  CS_HIP(hipSetDevice(p->device));
  if (!p->opt.use_graph) {
    CS_TRY(issue_steps(p, steps));
    p->steps_done += steps;
    return CS_OK;
  }
  // Graphs are keyed by (step count, starting buffer, fusion rule): the captured
  // kernel arguments name the buffers directly.
  const auto key = std::make_pair(steps * 4 + (p->halo_uniform ? 2 : 0), p->cur);
  auto it = p->graphs.find(key);
  if (it == p->graphs.end()) {
    const int cur0 = p->cur;
    const int64_t launches0 = p->launches;
    hipGraph_t graph = nullptr;
    CS_HIP(hipStreamBeginCapture(p->stream, hipStreamCaptureModeThreadLocal));
    cs_status st = issue_steps(p, steps);
    hipError_t e = hipStreamEndCapture(p->stream, &graph);
    p->cur = cur0;
    p->launches = launches0;
    if (st != CS_OK) {
      if (graph) (void)hipGraphDestroy(graph);
      return st;
    }
    CS_HIP(e);
    hipGraphExec_t exec = nullptr;
    hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    CS_HIP(ei);
    it = p->graphs.emplace(key, exec).first;
  }
  CS_HIP(hipGraphLaunch(it->second, p->stream));
  const int64_t n = count_launches(p, steps);
  p->cur = (int)((p->cur + n) & 1);
  p->launches += n;
  p->steps_done += steps;
  return CS_OK;
}

void destroy_graphs(cs_plan *p) {
  for (auto &kv : p->graphs) (void)hipGraphExecDestroy(kv.second);
  p->graphs.clear();
}

std::string tune_key(const cs_layout &L, int ndim, int R, int shape, const cs_options &o) {
  char k[160];
  snprintf(k, sizeof k, "d%d_r%d_s%d_p%d_n%lldx%lldx%lld_g%d_f%d", ndim, R, shape, o.precision, (long long)L.n[0],
           (long long)L.n[1], (long long)L.n[2], o.use_graph ? 1 : 0, o.fusion_depth);
  return std::string(k);
}

// Variants a plan may run: same radius and precision, its shape class (split precision:
// also the box variants), and the requested fusion depth if one is set.
std::vector<const Variant *> tune_candidates(const cs_plan *p, int classified_shape) {
  std::vector<const Variant *> out;
  int cnt = 0;
  const Variant *vs = family(p->ndim, &cnt, p->opt.precision);
  for (int i = 0; i < cnt; ++i) {
    const Variant &v = vs[i];
    if (v.R != p->R) continue;
    if (v.shape != classified_shape && !(p->opt.precision != CS_PREC_FP64 && v.shape == cs::SHAPE_BOX)) continue;
    if (p->opt.precision != CS_PREC_FP64 && v.mf != p->opt.precision) continue;
    // the --breakdown ladder's FMA kernels (for split plans mf holds the precision instead)
    if (p->opt.precision == CS_PREC_FP64 && (v.mf == 1 || v.mf == 2)) continue;
    if (p->opt.fusion_depth > 0 && v.kf != p->opt.fusion_depth) continue;
    if (p->ndim >= 2 && p->opt.precision == CS_PREC_FP64 &&
        (!fits(&v, p->L.n[1], p->L.n[2]) || (v.mf == 11 && p->L.n[1] * p->L.n[2] > 16000000)))
      continue;  // the register tiles are for small grids
    out.push_back(&v);
  }
  return out;
}

}  // namespace

extern "C" {

const char *cs_version(void) { return "convstencil-mi355x 0.1.0 (gfx950)"; }

const char *cs_status_string(cs_status s) {
  switch (s) {
    case CS_OK: return "ok";
    case CS_ERR_INVALID: return "invalid argument";
    case CS_ERR_UNSUPPORTED: return "unsupported configuration";
    case CS_ERR_ALLOC: return "allocation failed";
    case CS_ERR_DEVICE: return "HIP error";
    case CS_ERR_NO_DEVICE: return "no gfx950 device";
  }
  return "unknown status";
}

cs_status cs_device_count(int32_t *count) {
  if (!count) return CS_ERR_INVALID;
  *count = 0;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return CS_OK;
  for (int d = 0; d < n; ++d) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, d) == hipSuccess && strncmp(prop.gcnArchName, "gfx950", 6) == 0) ++*count;
  }
  return CS_OK;
}

void cs_fill_random_host(double *a, const cs_layout *L, uint64_t seed) {
  if (!a || !L) return;
  const int64_t total = cell_count(L);
  std::fill(a, a + total, 0.0);
  uint64_t st = cs::stream_seed(seed, 0);
  for (int64_t z = 0; z < L->n[0]; ++z)
    for (int64_t y = 0; y < L->n[1]; ++y) {
      double *row = a + ((L->org[0] + z) * L->ext[1] + (L->org[1] + y)) * L->ext[2] + L->org[2];
      for (int64_t x = 0; x < L->n[2]; ++x) row[x] = cs::unit_data(cs::splitmix_next(st));
    }
}

void cs_fill_weights_host(double *w, int32_t count, uint64_t seed) {
  if (!w || count <= 0) return;
  uint64_t st = cs::stream_seed(seed, 1);
  double s = 0.0;
  for (int i = 0; i < count; ++i) {
    w[i] = cs::unit_weight(cs::splitmix_next(st));
    s = s + w[i];
  }
  for (int i = 0; i < count; ++i) w[i] = w[i] / s;
}

}  // extern "C"

namespace {

// Times every candidate variant for at least kTuneSteps steps, a whole number of its
// fused launches (a remainder launch would come from another variant), with the graph
// as the plan asks, on the plan's own buffers and seeded synthetic data, and keeps the
// fastest -- unless it beats the library's default choice by less than kTuneMargin, a
// difference that timings on one device repeat within (box2d1r 10240^2: depth 8 and 12
// within 2%, picked either way run to run); the buffers are zeroed afterwards (the caller
// uploads or fills next).
constexpr int64_t kTuneSteps = 96;
constexpr double kTuneMargin = 0.03;

cs_status autotune_plan(cs_plan *p, int classified) {
  const std::vector<const Variant *> cand = tune_candidates(p, classified);
  if (cand.empty()) return CS_OK;
  const cs_options user = p->opt;
  int best = 0, dflt = 0;
  double best_ms = 1e300, dflt_ms = 1e300;
  p->shape = classified;
  if (select_variants(p) == CS_OK) dflt = p->vmain->id;
  for (const Variant *v : cand) {
    destroy_graphs(p);
    p->opt = user;
    p->opt.tile_variant = v->id;
    p->shape = classified;
    if (select_variants(p) != CS_OK) continue;
    CS_TRY(cs_plan_fill_random(p, 1));
    cs_report r{};
    const int64_t steps = (kTuneSteps + v->kf - 1) / v->kf * v->kf;
    CS_TRY(cs_plan_time(p, steps, 1, 3, &r));
    const double ms = r.elapsed_ms / (double)steps;
    if (p->opt.verbose) fprintf(stderr, "convstencil: autotune %s %.4f ms/step\n", v->name, ms);
    if (ms < best_ms) {
      best_ms = ms;
      best = v->id;
    }
    if (v->id == dflt) dflt_ms = ms;
  }
  if (dflt != 0 && best_ms > dflt_ms * (1.0 - kTuneMargin)) {
    best = dflt;
    best_ms = dflt_ms;
  }
  destroy_graphs(p);
  p->opt = user;
  p->shape = classified;
  if (best == 0) return select_variants(p);
  p->opt.tile_variant = best;
  CS_TRY(select_variants(p));
  p->tuned = 2;
  CS_HIP(cs::launch_zero(p->buf[0], (size_t)cell_count(&p->L), p->stream));
  CS_HIP(cs::launch_zero(p->buf[1], (size_t)cell_count(&p->L), p->stream));
  CS_HIP(hipStreamSynchronize(p->stream));
  p->cur = 0;
  p->steps_done = 0;
  p->halo_uniform = true;
  return cs_tune_store(tune_key(p->L, p->ndim, p->R, classified, user).c_str(), best, best_ms);
}

}  // namespace

namespace cs {

// A batch's launches of the register-streaming 2-D family for `steps` steps of a radius-R
// stencil of this shape class: the family's default depth as often as it fits, then its
// largest depth that fits the rest; empty where it has none.
void reg_sequence(int R, int shape, int64_t steps, std::vector<const Variant *> *seq) {
  seq->clear();
  const Variant *v = pick_main(2, R, shape, CS_PREC_FP64, 0, 0);  // no single grid: never mf 10
  if (!v || v->mf != 7) return;
  for (int64_t done = 0; done < steps;) {
    const int64_t rem = steps - done;
    const Variant *u = nullptr;
    if (rem >= v->kf) {
      u = v;
    } else {
      const int top = max_kf(2, 7, R, shape);  // the largest compiled depth that fits
      for (int kf = (int)std::min<int64_t>(rem, top); kf >= 1 && !u; --kf) u = find_variant(2, 7, R, shape, kf, 0);
    }
    if (!u) {
      seq->clear();
      return;
    }
    seq->push_back(u);
    done += u->kf;
  }
}

// The same for the register-tile kernels, for several grids of one stencil that share their launches
// (sizes: rows, columns), cut evenly, and its predicted time (*us): empty when there is no tile that
// fits them all.  The caller prepares them.
cs_status block_sequence(int R, int shape, const std::vector<std::pair<int64_t, int64_t>> &sizes, int64_t steps,
                         std::vector<const Variant *> *seq, double *us) {
  seq->clear();
  int cnt = 0;
  const Variant *vs = variants_2d_block(&cnt), *best = nullptr;
  double best_t = 1e300;
  for (int i = 0; i < cnt; ++i) {
    const Variant &v = vs[i];
    if (v.R != R || v.shape != shape || v.kf > steps) continue;
    const int64_t wo = v.bx - 2 * R * v.kf, to = v.by - 2 * R * v.kf;
    int64_t tiles = 0, edge = 0;
    double cells = 0.0;
    bool ok = !sizes.empty();
    for (const auto &n : sizes) {
      ok = ok && fits(&v, n.first, n.second);
      if (!ok) break;
      const int64_t tx = 1 + (n.second - v.bx + wo - 1) / wo, ty = 1 + (n.first - v.by + to - 1) / to;
      tiles += tx * ty;
      edge += std::min<int64_t>(tx, 2) * ty;
      cells += (double)n.first * (double)n.second;
    }
    if (!ok) continue;
    const double t = tiles_us_2d(v, tiles, edge, cells) / v.kf;
    if (t < best_t) {
      best_t = t;
      best = &v;
    }
  }
  if (!best) return CS_OK;
  *us = best_t * (double)steps;
  const int64_t n = (steps + best->kf - 1) / best->kf;
  for (int64_t i = 0; i < n; ++i) {
    const int64_t d = steps / n + (i < steps % n);
    const Variant *u = find_variant(2, 11, R, shape, (int)d, 0, CS_PREC_FP64, best->st);
    if (!u) return CS_ERR_UNSUPPORTED;
    seq->push_back(u);
  }
  return CS_OK;
}

// The FP64 kernel choice of a plan with a depth or a variant of its caller's, made without a plan (nothing
// allocated, no device touched): the main variant, the single-step variant and one variant per
// remainder depth 1 .. kf - 1 (vrem[r], null where the family has none), as select_variants picks them
// for a grid of ny x nx interior cells with a zero halo.
cs_status pick_fp64_variants(int ndim, int R, int shape, int fusion_depth, int tile_variant, int64_t ny, int64_t nx,
                             const Variant **vmain, const Variant **vone, const Variant **vrem, int vrem_cap) {
  const Variant *v = pick_main(ndim, R, shape, CS_PREC_FP64, fusion_depth, tile_variant, ny, nx);
  if (!v) return tile_variant > 0 ? CS_ERR_INVALID : CS_ERR_UNSUPPORTED;
  const Variant *strip = tile_variant <= 0 && ndim == 2 ? strip_of(v, fusion_depth, ny, nx) : nullptr;
  if (strip) v = strip;
  if (v->kf > vrem_cap) return CS_ERR_UNSUPPORTED;
  *vmain = v;
  *vone = single_step(ndim, R, v->shape, v);
  if (!*vone) return CS_ERR_UNSUPPORTED;
  for (int r = 0; r < vrem_cap; ++r)
    vrem[r] = r < 1 || r >= v->kf ? nullptr
              : strip             ? strip_remainder(strip, r)
                                  : remainder_variant(ndim, R, v->shape, v, r, CS_PREC_FP64, -1);
  return CS_OK;
}

}  // namespace cs

extern "C" {

cs_status cs_tune_key(const cs_layout *layout, const cs_stencil *st, const cs_options *opt, char *buf, int32_t len) {
  if (!layout || !st || !st->weights || !buf || len <= 0 || st->ndim != layout->ndim || st->radius < 1 ||
      st->radius > 4)
    return CS_ERR_INVALID;
  const int R = st->radius;
  const int shape = layout->ndim == 2 ? classify_2d(R, st->weights)
                    : layout->ndim == 3 ? classify_3d(R, st->weights)
                                        : cs::SHAPE_BOX;
  cs_options o{};
  if (opt) o = *opt;
  const std::string k = tune_key(*layout, layout->ndim, R, shape, o);
  if ((int32_t)k.size() >= len) return CS_ERR_INVALID;
  memcpy(buf, k.c_str(), k.size() + 1);
  return CS_OK;
}

cs_status cs_plan_create(cs_plan **out, const cs_layout *layout, const cs_stencil *st, const cs_options *opt) {
  if (!out || !layout || !st || !st->weights) return CS_ERR_INVALID;
  *out = nullptr;
  if (st->ndim != layout->ndim || st->radius < 1) return CS_ERR_INVALID;
  if (!layout_valid(layout, st->radius)) return CS_ERR_INVALID;
  if (st->radius > (st->ndim == 1 ? 4 : 3)) return CS_ERR_UNSUPPORTED;
  int dev = 0;
  CS_TRY(check_device(&dev));
  cs_plan *p = new cs_plan();
  p->L = *layout;
  p->ndim = layout->ndim;
  p->R = st->radius;
  const int D = 2 * p->R + 1;
  const int nw = p->ndim == 1 ? D : p->ndim == 2 ? D * D : D * D * D;
  p->w.assign(st->weights, st->weights + nw);
  if (opt) p->opt = *opt;
  p->device = dev;
  p->shape = p->ndim == 2 ? classify_2d(p->R, p->w.data()) : p->ndim == 3 ? classify_3d(p->R, p->w.data()) : cs::SHAPE_BOX;
  const int classified = p->shape;
  if (p->opt.autotune > 0 && p->opt.tile_variant == 0) {  // a cached choice needs no timing
    int32_t vid = 0;
    if (p->opt.autotune == 1 &&
        cs_tune_lookup(tune_key(p->L, p->ndim, p->R, classified, p->opt).c_str(), &vid, nullptr) == CS_OK) {
      p->opt.tile_variant = vid;
      p->tuned = 1;
    }
  }
  cs_status s = select_variants(p);
  if (s != CS_OK && p->tuned) {  // a stale cache entry: choose again
    p->opt.tile_variant = 0;
    p->tuned = 0;
    p->shape = classified;
    s = select_variants(p);
  }
  if (s != CS_OK) {
    cs_plan_destroy(p);
    return s;
  }
  if (hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking) != hipSuccess) {
    cs_plan_destroy(p);
    return CS_ERR_DEVICE;
  }
  const size_t bytes = (size_t)cell_count(layout) * sizeof(double);
  if (hipMalloc(&p->buf[0], bytes) != hipSuccess || hipMalloc(&p->buf[1], bytes) != hipSuccess) {
    (void)hipGetLastError();
    cs_plan_destroy(p);
    return CS_ERR_ALLOC;
  }
  // both buffers start at zero, so the range guard's bound (0) holds before any upload
  if (cs::launch_zero(p->buf[0], (size_t)cell_count(layout), p->stream) != hipSuccess ||
      cs::launch_zero(p->buf[1], (size_t)cell_count(layout), p->stream) != hipSuccess ||
      hipStreamSynchronize(p->stream) != hipSuccess) {
    cs_plan_destroy(p);
    return CS_ERR_DEVICE;
  }
  p->amax = 0.0;
  p->wabs = abs_sum(p->w.data(), p->w.size());
  if (p->opt.autotune > 0 && p->opt.tile_variant == 0) {
    s = autotune_plan(p, classified);
    if (s != CS_OK) {
      cs_plan_destroy(p);
      return s;
    }
  }
  *out = p;
  return CS_OK;
}

cs_status cs_plan_destroy(cs_plan *p) {
  if (!p) return CS_ERR_INVALID;
  if (p->stream) (void)hipStreamSynchronize(p->stream);
  destroy_graphs(p);
  for (double *&b : p->buf)
    if (b) (void)hipFree(b);
  if (p->bfrag) (void)hipFree(p->bfrag);
  if (p->stream) (void)hipStreamDestroy(p->stream);
  delete p;
  return CS_OK;
}

cs_status cs_plan_upload(cs_plan *p, const double *host_in) {
  if (!p || !host_in) return CS_ERR_INVALID;
  CS_HIP(hipSetDevice(p->device));
  const size_t n = (size_t)cell_count(&p->L);
  CS_HIP(hipMemcpyAsync(p->buf[0], host_in, n * sizeof(double), hipMemcpyHostToDevice, p->stream));
  CS_HIP(cs::launch_zero(p->buf[1], n, p->stream));
  CS_HIP(hipStreamSynchronize(p->stream));
  p->cur = 0;
  p->steps_done = 0;
  p->halo_uniform = halo_is_zero(&p->L, host_in);
  if (p->by_time && !p->halo_uniform) CS_TRY(prepare_sequence(p->seq[0]));
  // the scan (5.2 ms for 2048^2, of 11 ms for a whole host-to-host run) serves the FP16 range guard only
  p->amax = p->opt.precision == CS_PREC_FP16X2 || p->opt.precision == CS_PREC_FP16W3 ? abs_max(host_in, n) : 0.0;
  return CS_OK;
}

cs_status cs_plan_fill_random(cs_plan *p, uint64_t seed) {
  if (!p) return CS_ERR_INVALID;
  CS_HIP(hipSetDevice(p->device));
  Geo g{};
  for (int d = 0; d < 3; ++d) {
    g.ext[d] = p->L.ext[d];
    g.org[d] = p->L.org[d];
    g.n[d] = p->L.n[d];
  }
  CS_HIP(cs::launch_fill_random(p->buf[0], g, cs::stream_seed(seed, 0), p->stream));
  CS_HIP(cs::launch_zero(p->buf[1], (size_t)cell_count(&p->L), p->stream));
  CS_HIP(hipStreamSynchronize(p->stream));
  p->cur = 0;
  p->steps_done = 0;
  p->halo_uniform = true;
  p->amax = 1.0;  // the fill is uniform in [-1, 1) with a zero halo
  return CS_OK;
}

cs_status cs_plan_run(cs_plan *p, int64_t steps, cs_report *rep) {
  if (!p) return CS_ERR_INVALID;
  const int64_t l0 = p->launches;
  CS_TRY(run_steps(p, steps));
  if (rep) {
    memset(rep, 0, sizeof(*rep));
    rep->launches = p->launches - l0;
    rep->fusion_depth = executed_depth(p, steps);
    rep->variant = main_variant(p)->id;
  }
  return CS_OK;
}

cs_status cs_plan_time(cs_plan *p, int64_t steps, int32_t warmup, int32_t reps, cs_report *rep) {
  if (!p || reps <= 0 || warmup < 0 || steps <= 0) return CS_ERR_INVALID;
  CS_HIP(hipSetDevice(p->device));
  // graphs are captured per starting buffer: a run of an odd number of launches alternates
  // the two, so a warm-up captures both before the timed runs
  if (warmup > 0 && p->opt.use_graph && (count_launches(p, steps) & 1)) warmup = std::max(warmup, 2);
  for (int i = 0; i < warmup; ++i) CS_TRY(run_steps(p, steps));
  CS_HIP(hipStreamSynchronize(p->stream));
  hipEvent_t e0, e1;
  CS_HIP(hipEventCreate(&e0));
  CS_HIP(hipEventCreate(&e1));
  const int64_t l0 = p->launches;
  CS_HIP(hipEventRecord(e0, p->stream));
  for (int i = 0; i < reps; ++i) CS_TRY(run_steps(p, steps));
  CS_HIP(hipEventRecord(e1, p->stream));
  CS_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  CS_HIP(hipEventElapsedTime(&ms, e0, e1));
  CS_HIP(hipEventDestroy(e0));
  CS_HIP(hipEventDestroy(e1));
  if (rep) {
    memset(rep, 0, sizeof(*rep));
    rep->elapsed_ms = ms / reps;
    const double pts = (double)p->L.n[0] * (double)p->L.n[1] * (double)p->L.n[2];
    // a grid without interior cells launches nothing: no rate
    rep->gstencil_per_s = rep->elapsed_ms > 0 && pts > 0 ? pts * (double)steps / (rep->elapsed_ms * 1e-3) / 1e9 : 0.0;
    rep->launches = (p->launches - l0) / reps;
    rep->fusion_depth = executed_depth(p, steps);
    rep->variant = main_variant(p)->id;
  }
  return CS_OK;
}

cs_status cs_plan_sync(cs_plan *p) {
  if (!p) return CS_ERR_INVALID;
  CS_HIP(hipStreamSynchronize(p->stream));
  return CS_OK;
}

cs_status cs_plan_download(cs_plan *p, double *host_out) {
  if (!p || !host_out) return CS_ERR_INVALID;
  CS_HIP(hipSetDevice(p->device));
  CS_HIP(hipMemcpyAsync(host_out, p->buf[p->cur], (size_t)cell_count(&p->L) * sizeof(double), hipMemcpyDeviceToHost,
                        p->stream));
  CS_HIP(hipStreamSynchronize(p->stream));
  return CS_OK;
}

cs_status cs_plan_device_buffers(cs_plan *p, double **current, double **other) {
  if (!p) return CS_ERR_INVALID;
  if (current) *current = p->buf[p->cur];
  if (other) *other = p->buf[p->cur ^ 1];
  return CS_OK;
}

cs_status cs_plan_describe(cs_plan *p, char *buf, int32_t len) {
  if (!p || !buf || len <= 0) return CS_ERR_INVALID;
  static const char *how[3] = {"default", "cached", "timed"};
  const Variant *v = main_variant(p);
  snprintf(buf, (size_t)len,
           "variant=%d name=%s mf=%d R=%d shape=%s kf=%d tile=%dx%d waves=%d lds=%zu halo_uniform=%d autotune=%s",
           v->id, v->name, v->mf, p->R, p->shape == cs::SHAPE_BOX ? "box" : "star", v->kf, v->by, v->bx, v->nw, v->lds_bytes,
           (int)p->halo_uniform, how[p->tuned]);
  return CS_OK;
}

cs_status cs_run(const cs_layout *layout, const cs_stencil *st, const double *host_in, double *host_out, int64_t steps,
                 const cs_options *opt, cs_report *rep) {
  if (!host_in || !host_out || steps < 0) return CS_ERR_INVALID;
  cs_plan *p = nullptr;
  CS_TRY(cs_plan_create(&p, layout, st, opt));
  cs_status s = cs_plan_upload(p, host_in);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (s == CS_OK && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)) s = CS_ERR_DEVICE;
  if (s == CS_OK && hipEventRecord(e0, p->stream) != hipSuccess) s = CS_ERR_DEVICE;
  const int64_t l0 = p->launches;  // the autotuner's timing launches are not this run's
  if (s == CS_OK) s = run_steps(p, steps);
  if (s == CS_OK && hipEventRecord(e1, p->stream) != hipSuccess) s = CS_ERR_DEVICE;
  if (s == CS_OK) s = cs_plan_download(p, host_out);
  if (s == CS_OK && rep) {
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    memset(rep, 0, sizeof(*rep));
    rep->elapsed_ms = ms;
    const double pts = (double)layout->n[0] * (double)layout->n[1] * (double)layout->n[2];
    rep->gstencil_per_s = ms > 0 ? pts * (double)steps / (ms * 1e-3) / 1e9 : 0.0;
    rep->launches = p->launches - l0;
    rep->fusion_depth = executed_depth(p, steps);
    rep->variant = main_variant(p)->id;
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  cs_plan_destroy(p);
  return s;
}

}  // extern "C"
