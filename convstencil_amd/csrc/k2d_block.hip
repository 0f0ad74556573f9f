// k2d_block.hip -- FP64 2-D kernels that hold a whole tile in the registers of one workgroup
// (box and star of radius 1, star of radius 3), for grids that give a CU only a few thousand cells.
//
// Replaces kernel2d (reference src/2d/gpu.cu:30-70) and its time loop (src/2d/gpu.cu:316-329,
// 336-425) there.  The streaming kernels (k2d_reg.hip, k2d_pipe_body.h) sweep a chunk row after
// row and pay 2 R KF warm-up rows per chunk; on a small grid a chunk has fewer rows than that and
// its time is that chain's: 300 x 517 cells, box radius 1, 13 us for a launch of 4 steps.  Here a
// workgroup of 8 waves holds 32 or 64 rows of 128 columns (radius 3: 64 x 256) and advances them
// kf steps; what a step costs is its FMAs, two lane shifts per row and one exchange of the waves'
// outermost rows through LDS with a barrier.  Tiles overlap by 2 R kf cells.
//
// What bounds them: on the smallest grids the launch (about 4.5 us back to back in a graph) and
// the chain of steps, 0.55 us each (32 rows); on 2048^2 the FMAs, 1.5 times the useful ones for the
// overlap.  Measured, us per step, before (k2d_reg) and now: box radius 1 300 x 517 3.3 -> 1.0,
// 1024^2 4.6 -> 1.5, 1531 x 2749 5.8 -> 3.9, 2048^2 5.5 -> 3.9; star radius 1 300 x 517 2.4 -> 0.9,
// 2048^2 4.0 -> 3.0; star radius 3 512^2 7.4 -> 3.9, 1024^2 8.0 -> 4.3.  Shapes tried for the box: 256
// columns by 64 rows (4 per lane) 4.2 at 2048^2, 1024 threads 4.5-4.9; 16-row tiles 1.6 at 300 x 517.
//
// Halo: as in k2d_pipe_body.h.  The first tile starts at cell 0, the last ends at cell n - 1 of
// each axis (where the last two overlap further both store the same bits); +0 halos come from the
// lane shifts' zero fill and zeroed rows, others are read from memory per step, from the buffer
// that the step of the ping-pong reads (Geo::flip exchanges them).
#include "cs_internal.h"

namespace cs {

namespace {

typedef const double __attribute__((address_space(4))) cdouble;  // scalar loads
typedef const double __attribute__((address_space(1))) gdouble;
typedef const RegItem __attribute__((address_space(4))) citem;
typedef const RegGrid __attribute__((address_space(4))) cgrid;
typedef double pair_t __attribute__((ext_vector_type(2)));

struct BlockSplit {
  int tx, ty, kf;
};

__device__ __forceinline__ double lower_or(double v, double f) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(f), __double2loint(v), 0x138, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(f), __double2hiint(v), 0x138, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double upper_or(double v, double f) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(f), __double2loint(v), 0x130, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(f), __double2hiint(v), 0x130, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ uint64_t opaque(const void *p) {
  const uint64_t v = (uint64_t)p;
  uint64_t u = (uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)v) |
               ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32);
  asm volatile("" : "+s"(u));
  return u;
}

// A tile of TR x W cells: wave w holds rows w BR .. w BR + BR - 1, lane l columns l PX ..
// l PX + PX - 1.
template <int R, int PX, int BR, int NWV>
struct Block2D {
  static constexpr int W = 64 * PX, TR = NWV * BR;
  static constexpr int PP = PX / 2;            // 16-byte pieces per lane and row
  static constexpr int SH = NWV * 2 * R * W;   // doubles shared per step: R rows at either end of every wave's
  static constexpr int NBUF = R == 1 ? 2 : 1;  // shared buffers; with one, a second barrier per step
  static constexpr int LDS = NBUF * SH;
  static_assert(R <= PX && R <= BR && PX % 2 == 0, "rows and lanes reach their neighbours only");
};

template <int R, int SHAPE, int PX, int BR, int NWV, bool GEN>
struct BlockRun {
  using C = Block2D<R, PX, BR, NWV>;
  static constexpr int D = 2 * R + 1, PP = C::PP;
  static constexpr bool BOX = SHAPE == SHAPE_BOX;
  static constexpr int RW = C::W / 2, WV = 2 * R * RW;  // pairs per shared row, per wave

  const double *in;
  double *out;
  double w[D * D];
  int64_t pitch, ey, oy, ox, nx, xs, row0;
  bool top, bottom;
  int flip, lane, wv;
  pair_t *sh;

  // Row i of the wave's tile rows in step s: its own, or (i < 0, i >= BR) one of the wave above's
  // last or below's first R rows.  Beyond the tile lies the halo, or, inside the grid, anything
  // (zero here): those cells' results reach no output.
  __device__ __forceinline__ void row(const double (&a)[BR][PX], int i, const pair_t *buf, const double *hb,
                                      double (&q)[PX]) {
    if (i >= 0 && i < BR) {
#pragma unroll
      for (int j = 0; j < PX; ++j) q[j] = a[i][j];
    } else if (i < 0 ? wv > 0 : wv < NWV - 1) {  // wave-uniform
      const pair_t *p = buf + (i < 0 ? (wv - 1) * WV + (2 * R + i) * RW : (wv + 1) * WV + (i - BR) * RW);
#pragma unroll
      for (int n = 0; n < PP; ++n) {
        const pair_t v = p[n * 64];
        q[2 * n] = v.x;
        q[2 * n + 1] = v.y;
      }
    } else {
#pragma unroll
      for (int j = 0; j < PX; ++j) q[j] = 0.0;
      if constexpr (GEN) {
        if (i < 0 ? top : bottom) {
          gdouble *p = (gdouble *)opaque(hb + (oy + row0 + i) * pitch + ox + xs);
#pragma unroll
          for (int j = 0; j < PX; ++j) q[j] = p[lane * PX + j];
        }
      }
    }
  }

  // One step from a to b; b's rows are their own accumulators (a chain of FMAs, rows dy = -R .. R,
  // columns dx = -R .. R, as in the other FP64 kernels).
  __device__ __forceinline__ void step(const double (&a)[BR][PX], double (&b)[BR][PX], int s) {
    pair_t *buf = sh + (C::NBUF == 2 ? (s & 1) * (C::SH / 2) : 0);
#pragma unroll
    for (int k = 0; k < R; ++k) {
#pragma unroll
      for (int i = 0; i < PP; ++i) {
        pair_t v;
        v.x = a[k][2 * i];
        v.y = a[k][2 * i + 1];
        buf[wv * WV + k * RW + i * 64] = v;
        v.x = a[BR - R + k][2 * i];
        v.y = a[BR - R + k][2 * i + 1];
        buf[wv * WV + (R + k) * RW + i * 64] = v;
      }
    }
    lds_barrier();
    // the buffer whose halo this step reads; a choice between copies, as in k2d_pipe_body.h (halo_buffer)
    const double *const even = in, *const odd = out;
    const double *hb = ((s + flip) & 1) ? odd : even;
#pragma unroll
    for (int i = -R; i < BR + R; ++i) {
      double q[PX], qe[PX + 2 * R];
      row(a, i, buf, hb, q);
#pragma unroll
      for (int j = 0; j < PX; ++j) qe[R + j] = q[j];
      if (BOX || (i >= 0 && i < BR)) {
        if constexpr (GEN) {
          int64_t ay = oy + row0 + i;
          ay = ay < 0 ? 0 : ay >= ey ? ey - 1 : ay;
          cdouble *h = (cdouble *)opaque(hb + ay * pitch + ox);
#pragma unroll
          for (int k = 0; k < R; ++k) {
            qe[k] = lower_or(q[PX - R + k], h[k - R]);
            qe[PX + R + k] = upper_or(q[k], h[nx + k]);
          }
        } else {
#pragma unroll
          for (int k = 0; k < R; ++k) {
            qe[k] = lane_from_lower(q[PX - R + k]);
            qe[PX + R + k] = lane_from_upper(q[k]);
          }
        }
      }
#pragma unroll
      for (int dy = R; dy >= -R; --dy) {
        const int t = i - dy;  // the output row that row i lies at offset dy of
        if (t < 0 || t >= BR) continue;
#pragma unroll
        for (int dx = -R; dx <= R; ++dx) {
          if (!BOX && dy != 0 && dx != 0) continue;
          const bool first = dy == -R && (BOX ? dx == -R : dx == 0);
#pragma unroll
          for (int j = 0; j < PX; ++j) {
            const double wt = w[(dy + R) * D + dx + R], v = qe[R + j + dx];
            b[t][j] = first ? wt * v : __builtin_fma(wt, v, b[t][j]);
          }
        }
      }
    }
    if constexpr (C::NBUF == 1) lds_barrier();  // every wave has read its neighbours' rows
  }

  __device__ __forceinline__ void run(int kf, int64_t ys, bool left, bool right) {
    double a[BR][PX], b[BR][PX];
    const double *src = in + (oy + row0) * pitch + ox + xs + lane * PX;
#pragma unroll
    for (int i = 0; i < BR; ++i)
#pragma unroll
      for (int j = 0; j < PX; ++j) a[i][j] = src[i * pitch + j];
    int s = 0;
    for (; s + 1 < kf; s += 2) {
      step(a, b, s);
      step(b, a, s + 1);
    }
    if (s < kf) {
      step(a, b, s);
#pragma unroll
      for (int i = 0; i < BR; ++i)
#pragma unroll
        for (int j = 0; j < PX; ++j) a[i][j] = b[i][j];
    }
    const int H = R * kf;
    const int lo = top ? 0 : H, hi = bottom ? C::TR : C::TR - H;
    const int cl = left ? 0 : H, ch = right ? C::W : C::W - H;
    double *dst = out + (oy + row0) * pitch + ox + xs + lane * PX;
#pragma unroll
    for (int i = 0; i < BR; ++i) {
      const int r = wv * BR + i;
      if (r < lo || r >= hi) continue;  // wave-uniform
#pragma unroll
      for (int j = 0; j < PX; ++j) {
        const int c = lane * PX + j;
        if (c >= cl && c < ch) dst[i * pitch + j] = a[i][j];
      }
    }
  }
};

template <int R, int SHAPE, int PX, int BR, int NWV, bool GEN>
__device__ __forceinline__ void run_block(const double *in, double *out, const double *wts, const Geo &g, int kf,
                                          int64_t xs, int64_t ys, bool left, bool right, bool top, bool bottom,
                                          int lane, int wv, double *lds) {
  BlockRun<R, SHAPE, PX, BR, NWV, GEN> t;
  t.in = in;
  t.out = out;
#pragma unroll
  for (int i = 0; i < t.D * t.D; ++i) t.w[i] = ((cdouble *)opaque(wts))[i];
  t.pitch = g.ext[2];
  t.ey = g.ext[1];
  t.oy = g.org[1];
  t.ox = g.org[2];
  t.nx = g.n[2];
  t.xs = xs;
  t.row0 = ys + wv * BR;
  t.top = top;
  t.bottom = bottom;
  t.flip = (int)g.flip;
  t.lane = lane;
  t.wv = wv;
  t.sh = (pair_t *)lds + lane;
  t.run(kf, ys, left, right);
}

extern __shared__ __attribute__((aligned(16))) double block_lds[];

// Tile (by, bx) of a grid by kf steps; right, bottom: the last one of its axis.
template <int R, int SHAPE, int PX, int BR, int NWV>
__device__ __forceinline__ void block_tile(const double *in, double *out, const double *wts, const Geo &g, int kf,
                                           int bx, int by, bool right, bool bottom) {
  using C = Block2D<R, PX, BR, NWV>;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = R * kf;
  const int64_t ny = g.n[1], nx = g.n[2], pitch = g.ext[2];
  const bool left = bx == 0, top = by == 0;
  const int64_t xs = right ? nx - C::W : (int64_t)bx * (C::W - 2 * H);
  const int64_t ys = bottom ? ny - C::TR : (int64_t)by * (C::TR - 2 * H);
  bool general = false;
  if (left || right || top || bottom) {
    const int64_t ya = top ? -R : ys, yb = bottom ? ny + R : ys + C::TR;
    uint64_t any = 0;
#pragma unroll 1
    for (int b = 0; b < 2; ++b) {
      const double *p = (b ? (const double *)out : in) + g.org[1] * pitch + g.org[2];
      if (left || right) {
        for (int64_t y = ya + threadIdx.x; y < yb; y += NWV * 64) {
#pragma unroll
          for (int k = 0; k < R; ++k) {
            if (left) any |= (uint64_t)__double_as_longlong(p[y * pitch - R + k]);
            if (right) any |= (uint64_t)__double_as_longlong(p[y * pitch + nx + k]);
          }
        }
      }
      for (int k = 0; k < R; ++k) {
        for (int64_t x = xs + threadIdx.x; x < xs + C::W; x += NWV * 64) {
          if (top) any |= (uint64_t)__double_as_longlong(p[(k - R) * pitch + x]);
          if (bottom) any |= (uint64_t)__double_as_longlong(p[(ny + k) * pitch + x]);
        }
      }
    }
    general = __syncthreads_or(any != 0);
  }
  if (general)
    run_block<R, SHAPE, PX, BR, NWV, true>(in, out, wts, g, kf, xs, ys, left, right, top, bottom, lane, wv, block_lds);
  else
    run_block<R, SHAPE, PX, BR, NWV, false>(in, out, wts, g, kf, xs, ys, left, right, top, bottom, lane, wv,
                                            block_lds);
}

template <int R, int SHAPE, int PX, int BR, int NWV>
__global__ __launch_bounds__(NWV * 64, R == 1 ? 4 : 2) void k2d_block(const double *in, double *out, const double *wts, Geo g,
                                                     BlockSplit sp) {
  const int by = __builtin_amdgcn_readfirstlane(blockIdx.x / (unsigned)sp.tx);
  const int bx = (int)blockIdx.x - by * sp.tx;
  block_tile<R, SHAPE, PX, BR, NWV>(in, out, wts, g, sp.kf, bx, by, bx == sp.tx - 1, by == sp.ty - 1);
}

// The tiles of several grids: item.strip, item.y0 = bx, by; item.y1 = right | bottom << 1.
template <int R, int SHAPE, int PX, int BR, int NWV>
__global__ __launch_bounds__(NWV * 64, R == 1 ? 4 : 2) void k2d_block_multi(RegMulti mm, int kf) {
  // item, grid and weights by scalar loads: they are the workgroup's, and as vectors they spill (radius
  // 3: 66 registers)
  const citem *it = (citem *)opaque(mm.items + blockIdx.x);
  const cgrid *G = (cgrid *)opaque(mm.grids + it->grid);
  const int cur = G->cur ^ mm.flip, y1 = it->y1;
  Geo g;
  for (int d = 0; d < 3; ++d) {
    g.ext[d] = G->geo.ext[d];
    g.org[d] = G->geo.org[d];
    g.n[d] = G->geo.n[d];
  }
  g.flip = G->geo.flip;
  const double *const b0 = G->buf[0], *const b1 = G->buf[1];
  block_tile<R, SHAPE, PX, BR, NWV>(cur ? b1 : b0, (double *)(cur ? b0 : b1), G->wts, g, kf, it->strip, it->y0, y1 & 1,
                                    y1 >> 1);
}

template <int R, int SHAPE, int PX, int BR, int NWV>
struct BlockLaunch {
  using C = Block2D<R, PX, BR, NWV>;
  static constexpr size_t kLds = C::LDS * sizeof(double);

  static hipError_t prepare() {
    hipError_t e = hipFuncSetAttribute((const void *)k2d_block<R, SHAPE, PX, BR, NWV>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
    if (e != hipSuccess) return e;
    return hipFuncSetAttribute((const void *)k2d_block_multi<R, SHAPE, PX, BR, NWV>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
  }

  template <int KF>
  static hipError_t launch_multi(const RegMulti &mm, hipStream_t s) {
    hipLaunchKernelGGL((k2d_block_multi<R, SHAPE, PX, BR, NWV>), dim3((unsigned)mm.nitems), dim3(NWV * 64), kLds, s, mm,
                       KF);
    return hipGetLastError();
  }

  template <int KF>
  static hipError_t launch(const double *in, double *out, const double *wts, const Geo &g, hipStream_t s) {
    const int64_t ny = g.n[1], nx = g.n[2], wo = C::W - 2 * R * KF, to = C::TR - 2 * R * KF;
    if (nx < C::W || ny < C::TR) return hipErrorInvalidValue;
    const int64_t tx = 1 + (nx - C::W + wo - 1) / wo, ty = 1 + (ny - C::TR + to - 1) / to;
    if (tx * ty > 0x7fffffff) return hipErrorInvalidValue;
    const BlockSplit sp{(int)tx, (int)ty, KF};
    hipLaunchKernelGGL((k2d_block<R, SHAPE, PX, BR, NWV>), dim3((unsigned)(tx * ty)), dim3(NWV * 64), kLds, s, in, out,
                       wts, g, sp);
    return hipGetLastError();
  }
};

}  // namespace

// Variant::mf 11 marks this family: by x bx = the tile, px = columns per lane, st = rows per wave;
// one kernel serves every depth.
#define CS_VB2D(ID, R, SH, PX, BR, NWV, KF)                                                                  \
  Variant {                                                                                                  \
    ID + KF, 11, R, SH, KF, NWV *BR, 64 * PX, NWV, BlockLaunch<R, SH, PX, BR, NWV>::kLds, PX, BR,            \
        &BlockLaunch<R, SH, PX, BR, NWV>::launch<KF>, &BlockLaunch<R, SH, PX, BR, NWV>::prepare,             \
        "k2d_block<r" #R "," #SH ",p" #PX "," #BR "x" #NWV ",kf" #KF ">",                                    \
        0, &BlockLaunch<R, SH, PX, BR, NWV>::launch_multi<KF>                                                \
  }
#define CS_VB2D7(ID, R, SH, PX, BR, NWV)                                            \
  CS_VB2D(ID, R, SH, PX, BR, NWV, 1), CS_VB2D(ID, R, SH, PX, BR, NWV, 2),           \
      CS_VB2D(ID, R, SH, PX, BR, NWV, 3), CS_VB2D(ID, R, SH, PX, BR, NWV, 4),       \
      CS_VB2D(ID, R, SH, PX, BR, NWV, 5), CS_VB2D(ID, R, SH, PX, BR, NWV, 6),       \
      CS_VB2D(ID, R, SH, PX, BR, NWV, 7)
#define CS_VB2D12(ID, R, SH, PX, BR, NWV)                                           \
  CS_VB2D7(ID, R, SH, PX, BR, NWV), CS_VB2D(ID, R, SH, PX, BR, NWV, 8),             \
      CS_VB2D(ID, R, SH, PX, BR, NWV, 9), CS_VB2D(ID, R, SH, PX, BR, NWV, 10),      \
      CS_VB2D(ID, R, SH, PX, BR, NWV, 11), CS_VB2D(ID, R, SH, PX, BR, NWV, 12)

// ids 2000000 + (star) * 100000 + R * 10000 + BR * 100 + KF
static const Variant kVariantsBlock2D[] = {
    CS_VB2D12(2010400, 1, SHAPE_BOX, 2, 4, 8),
    CS_VB2D12(2010800, 1, SHAPE_BOX, 2, 8, 8),
    CS_VB2D12(2110400, 1, SHAPE_STAR, 2, 4, 8),
    CS_VB2D12(2110800, 1, SHAPE_STAR, 2, 8, 8),
    CS_VB2D7(2130800, 3, SHAPE_STAR, 4, 8, 8),
};

const Variant *variants_2d_block(int *count) {
  *count = (int)(sizeof(kVariantsBlock2D) / sizeof(kVariantsBlock2D[0]));
  return kVariantsBlock2D;
}

}  // namespace cs
