// k3d_tile.hip -- z-streaming FP64 3-D kernels of radius 1 (27-point box, 7-point star): a
// workgroup's waves stack into one tall tile and exchange their border rows through LDS.
//
// Replaces gpu_box_3d1r_kernel and gpu_star_3d1r_step3_kernel (reference
// src/3d/gpu_box.cu:186-238, src/3d/gpu_star.cu) for KF fused steps.  In k3d_reg.hip every wave is a tile of its own and
// recomputes 2 (KF - l) rows of level l around its 7 or 8 output rows, which ends at two (box) or three
// (star) steps.  Here 8 or 16 waves form a tile of up to 80 rows x 64 columns that streams its
// z range: rows are shared between the waves, so only the tile's own border of KF cells is
// recomputed and four steps pay.  Every iteration each level takes one plane and completes the one
// before it; a level reads what the level below completed an iteration earlier, so one barrier
// and two shared rows per wave and level serve all levels, and the levels, taken from the
// last to the first, need no copy of a completed plane.
//
// Halo (zero; plans with other halos take single steps): the first tile of an axis starts at
// the interior's first cell and the last ends at its last one, so the cells outside are the
// lane shifts' missing sources (zero), shared rows that are never written (zero) and planes
// that are set to zero; no row or column is masked.
//
// What bounds them (profiles/fp64_pipe_tile_counters.md): 512^3 box, 80 x 64 tiles at depth 3: FP64 issue (87% of
// the cycles, 43 TFLOP/s; a 27-tap row costs 27 FMAs and 5 lane-shift moves a cell, the overlap 1.19
// times the cells of a plane); star, 64 x 64 at depth 4: memory, 5.1 TB/s with the overlap's reads; small grids: the
// launch and the chain of planes.  Measured, us
// per step, k3d_reg's choice before and now: box 512^3 307 -> 211, 389 x 301 x 517 160 -> 105, 256^3
// 48 -> 41, 100^3 23.0 -> 8.4, 600 x 64 x 64 19.9 -> 10.9; star 512^3 211 -> 115, 389 x 301 x 517
// 92 -> 66, 256^3 30.7 -> 23.3, 100^3 11.1 -> 5.9.  Load rings of 2 or 3 planes instead of 1 gave nothing
// (star depth 3 174 and 172 against 173), five and six steps lose to four (star 389 x 301 x 517 77
// against 66).
#include <algorithm>

#include "cs_internal.h"

namespace cs {

namespace {

typedef const double __attribute__((address_space(1))) gdouble;

// A wave-uniform address in scalar registers, so that a load needs the lane's offset only.
__device__ __forceinline__ uint64_t opaque(const double *p) {
  const uint64_t v = (uint64_t)p;
  uint64_t u = (uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)v) |
               ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32);
  asm volatile("" : "+s"(u));
  return u;
}

// A tile of TY x 64 cells of every plane: wave w holds rows w RY .. w RY + RY - 1, lane l column l.
template <int RY, int KF, int NW>
struct Tile3D {
  static constexpr int TY = RY * NW, OX = 64 - 2 * KF, OY = TY - 2 * KF;
  // shared rows: [iteration parity][level 1 .. KF - 1][wave + 1][first, last][lane]; the first and
  // last entry of the third index stay zero (the halo above and below the tile)
  static constexpr int LV = (NW + 2) * 2 * 64, SH = (KF > 1 ? KF - 1 : 1) * LV;
  static constexpr int LDS = KF > 1 ? 2 * SH : 1;
};

struct Tile3Split {
  int tx, ty, zchunks, zc;
};

template <int SH, int RY, int KF, int NW, int RING>
struct Tile3Run {
  using C = Tile3D<RY, KF, NW>;
  static constexpr bool BOX = SH == SHAPE3_BOX;
  static constexpr int PER = RING % 3 == 0 ? RING : 3 * RING;
  static constexpr int NR = RY + 2;

  const double *in;  // the wave's row -1, column 0 of the tile, of plane 0
  double *out;       // the wave's row 0, column 0 of the tile, of plane 0
  double w[27];
  int64_t plane, ex;  // doubles per plane and row
  int nz, lane, wv, r0, r1;  // output rows r0 <= i < r1 of the wave
  int off;                   // the lane's store offset, or past the range where it has no output
  double *sh;                // the wave's rows of level 1, parity 0, this lane's entry
  double ring[RING][NR];
  double a[KF][3][RY];  // partial planes of level l + 1; plane q in slot (q - first plane) mod 3

  // Plane z, clamped to the halo planes next to the interior (zero, as every plane beyond).
  __device__ __forceinline__ void load(int z, double (&q)[NR]) {
    const int cz = z < -1 ? -1 : z > nz ? nz : z;
    const double *p = in + cz * plane;
#pragma unroll
    for (int r = 0; r < NR; ++r) q[r] = ((gdouble *)opaque(p + r * ex))[(unsigned)lane];
  }

  // Source row r (the wave's row r - 1) adds its taps to the rows r - 2 .. r of the planes
  // p - 1 (U, then complete), p (V) and p + 1 (T, started here).  Sum order per output: dz, dy, dx
  // ascending.
  __device__ __forceinline__ void row(double v, int r, double (&U)[RY], double (&V)[RY], double (&T)[RY]) {
    double lo = 0.0, hi = 0.0;
    asm volatile("" : "+v"(v));
    if (BOX || (r >= 1 && r <= RY)) {
      lo = lane_from_lower(v);
      hi = lane_from_upper(v);
    }
#pragma unroll
    for (int dy = -1; dy <= 1; ++dy) {
      const int i = r - 1 - dy;
      if (i < 0 || i >= RY) continue;
#pragma unroll
      for (int dz = 1; dz >= -1; --dz) {
        double(&A)[RY] = dz == 1 ? U : dz == 0 ? V : T;
        const double *c = w + ((dz + 1) * 3 + dy + 1) * 3;
        if (BOX) {
          A[i] = dz == -1 && dy == -1 ? c[0] * lo : __builtin_fma(c[0], lo, A[i]);
          A[i] = __builtin_fma(c[1], v, A[i]);
          A[i] = __builtin_fma(c[2], hi, A[i]);
        } else if (dz != 0) {
          if (dy == 0) A[i] = dz == -1 ? c[1] * v : __builtin_fma(c[1], v, A[i]);
        } else if (dy != 0) {
          A[i] = __builtin_fma(c[1], v, A[i]);
        } else {
          A[i] = __builtin_fma(c[0], lo, A[i]);
          A[i] = __builtin_fma(c[1], v, A[i]);
          A[i] = __builtin_fma(c[2], hi, A[i]);
        }
        asm volatile("" : "+v"(A[i]));
      }
    }
  }

  // Level L takes plane p = t - 2 (L - 1), which level L - 1 completed one iteration ago.
  template <int K, int L>
  __device__ __forceinline__ void level(int t, int z0, int z1, const double (&nb)[KF][2]) {
    constexpr int S = K - 2 * (L - 1) + 12;
    double(&U)[RY] = a[L - 1][(S - 1) % 3];
    double(&V)[RY] = a[L - 1][S % 3];
    double(&T)[RY] = a[L - 1][(S + 1) % 3];
    if constexpr (L == 1) {
      double(&q)[NR] = ring[K % RING];
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        row(q[r], r, U, V, T);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_sched_barrier(0);
      load(t + RING, q);
    } else {
      const double(&q)[RY] = a[L - 2][S % 3];
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        row(r == 0 ? nb[L - 1][0] : r == NR - 1 ? nb[L - 1][1] : q[r - 1], r, U, V, T);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // plane p - 1 is complete
    const int z = t - 2 * (L - 1) - 1;
    if constexpr (L < KF) {
      if (z < 0 || z >= nz) {  // the halo of an intermediate step
#pragma unroll
        for (int i = 0; i < RY; ++i) U[i] = 0.0;
      }
      double *p = sh + (K & 1) * C::SH + (L - 1) * C::LV;
      p[0] = U[0];
      p[64] = U[RY - 1];
    } else {
      const bool ok = z >= z0 && z < z1;
#pragma unroll
      for (int i = 0; i < RY; ++i) {
        const __amdgpu_buffer_rsrc_t rs =
            buffer_over(out + z * plane + i * ex, ok && i >= r0 && i < r1 ? 64 * 8 : 0);
        buffer_store1(rs, off, U[i]);
      }
    }
    if constexpr (L > 1) {
      __builtin_amdgcn_sched_barrier(0);
      level<K, L - 1>(t, z0, z1, nb);
    }
  }

  template <int K>
  __device__ __forceinline__ void phases(int t, int t1, int z0, int z1) {
    if constexpr (K < 2 * PER) {
      if (K == PER && t + K >= t1) return;  // the same for all waves
      double nb[KF][2];
#pragma unroll
      for (int l = 1; l < KF; ++l) {
        const double *p = sh + ((K + 1) & 1) * C::SH + (l - 1) * C::LV;
        nb[l][0] = p[-64];   // the wave above's last row
        nb[l][1] = p[128];   // the wave below's first row
      }
      level<K, KF>(t + K, z0, z1, nb);
      if constexpr (KF > 1) lds_barrier();
      phases<K + 1>(t, t1, z0, z1);
    }
  }

  __device__ __forceinline__ void run(int z0, int z1) {
#pragma unroll
    for (int l = 0; l < KF; ++l)
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int i = 0; i < RY; ++i) a[l][k][i] = 0.0;
    const int t0 = z0 - KF, t1 = z1 + 2 * KF - 1;
#pragma unroll
    for (int k = 0; k < RING; ++k) load(t0 + k, ring[k]);
    for (int t = t0; t < t1; t += 2 * PER) phases<0>(t, t1, z0, z1);
  }
};

template <int SH, int RY, int KF, int NW, int RING, int WPE>
__global__ __launch_bounds__(NW * 64, WPE) void k3d_tile(const double *__restrict__ in, double *__restrict__ out,
                                                         const double *__restrict__ wts, Geo g, Tile3Split sp) {
  using C = Tile3D<RY, KF, NW>;
  __shared__ double sh[C::LDS];
  // workgroups are dealt to the 8 XCDs in turn: each XCD takes a run of neighbouring tiles, whose
  // overlaps its L2 then holds (star, 512^3, depth 4: 142 -> 131 us a step)
  const int per = gridDim.x / 8, bx = blockIdx.x, b = bx < per * 8 ? bx % 8 * per + bx / 8 : bx;
  const int tile = b % (sp.tx * sp.ty);
  const int z0 = b / (sp.tx * sp.ty) * sp.zc, sx = tile % sp.tx, sy = tile / sp.tx;
  if constexpr (KF > 1) {
    for (int i = threadIdx.x; i < C::LDS; i += NW * 64) sh[i] = 0.0;
    lds_barrier();
  }
  Tile3Run<SH, RY, KF, NW, RING> S;
  S.lane = threadIdx.x & 63;
  S.wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  S.nz = (int)g.n[0];
  S.plane = g.ext[1] * g.ext[2];
  S.ex = g.ext[2];
  // the last tile of an axis ends with the grid; where it overlaps the one before by more than
  // 2 KF cells both store the same bits
  const int64_t xs = sx == sp.tx - 1 ? g.n[2] - 64 : (int64_t)sx * C::OX;
  const int64_t ys = sy == sp.ty - 1 ? g.n[1] - C::TY : (int64_t)sy * C::OY;
  const int64_t base = (g.org[0] * g.ext[1] + g.org[1] + ys + S.wv * RY) * S.ex + g.org[2] + xs;
  S.in = in + base - S.ex;
  S.out = out + base;
  S.r0 = (sy == 0 ? 0 : KF) - S.wv * RY;
  S.r1 = (sy == sp.ty - 1 ? C::TY : C::TY - KF) - S.wv * RY;
  S.off = S.lane >= (sx == 0 ? 0 : KF) && S.lane < (sx == sp.tx - 1 ? 64 : 64 - KF) ? S.lane * 8 : kBufferDrop;
  S.sh = sh + (KF > 1 ? (S.wv + 1) * 128 + S.lane : 0);
#pragma unroll
  for (int i = 0; i < 27; ++i) S.w[i] = wts[i];
  const int z1 = z0 + sp.zc < S.nz ? z0 + sp.zc : S.nz;
  S.run(z0, z1);
}

hipError_t prepare_tile3() { return hipSuccess; }

// Resident workgroups on 256 CUs.
constexpr int slots_of(int nw, int wpe) { return 256 * wpe * 4 / nw; }

// Tiles and z chunks of a launch: of 1 .. 64 chunks the count with the least rounds x iterations
// (every chunk pays 3 kf - 1 iterations before its last plane is out).
Tile3Split tile3_split(int64_t nz, int64_t ny, int64_t nx, int ty, int kf, int slots) {
  Tile3Split sp{};
  const int64_t ox = 64 - 2 * kf, oy = ty - 2 * kf;
  sp.tx = (int)(1 + (nx - 64 + ox - 1) / ox);
  sp.ty = (int)(1 + (ny - ty + oy - 1) / oy);
  const int64_t tiles = (int64_t)sp.tx * sp.ty;
  int64_t best = 0;
  for (int64_t c = 1; c <= nz && c <= 64; ++c) {
    const int64_t zc = (nz + c - 1) / c, n = (nz + zc - 1) / zc;
    const int64_t cost = (tiles * n + slots - 1) / slots * (zc + 3 * kf - 1);
    if (best == 0 || cost < best) {
      best = cost;
      sp.zc = (int)zc;
      sp.zchunks = (int)n;
    }
  }
  return sp;
}

template <int SH, int RY, int KF, int NW, int RING, int WPE>
hipError_t launch_tile3(const double *in, double *out, const double *wts, const Geo &g, hipStream_t s) {
  using C = Tile3D<RY, KF, NW>;
  if (g.n[2] < 64 || g.n[1] < C::TY || g.n[0] < 1 || g.n[0] > (1 << 30)) return hipErrorInvalidValue;
  const Tile3Split sp = tile3_split(g.n[0], g.n[1], g.n[2], C::TY, KF, slots_of(NW, WPE));
  hipLaunchKernelGGL((k3d_tile<SH, RY, KF, NW, RING, WPE>), dim3((unsigned)(sp.tx * sp.ty * sp.zchunks)),
                     dim3(NW * 64), 0, s, in, out, wts, g, sp);
  return hipGetLastError();
}

}  // namespace

// Variant::mf 12 marks this family: by x bx = the tile, halo included, nw = waves; st = planes in the
// load ring.  ids 4000000 + (star) * 100000 + waves * 1000 + rows per wave * 100 + steps * 10 + ring
#define CS_VT3(SH, RY, KF, NW, RING, WPE)                                                                   \
  Variant {                                                                                                 \
    4000000 + (SH == SHAPE3_STAR) * 100000 + NW * 1000 + RY * 100 + KF * 10 + RING, 12, 1, SH, KF, RY * NW, \
        64, NW, 0, 1, RING, &launch_tile3<SH, RY, KF, NW, RING, WPE>,                                       \
        &prepare_tile3,                                                                                     \
        "k3d_tile<r1," #SH ",ry" #RY ",kf" #KF ",w" #NW ",ring" #RING ",wpe" #WPE ">"                       \
  }

static const Variant kVariantsTile3D[] = {
    CS_VT3(SHAPE3_BOX, 8, 4, 8, 1, 2),   CS_VT3(SHAPE3_BOX, 8, 3, 8, 1, 2),   CS_VT3(SHAPE3_BOX, 8, 2, 8, 1, 2),
    CS_VT3(SHAPE3_BOX, 5, 3, 16, 1, 4),  CS_VT3(SHAPE3_BOX, 5, 2, 16, 1, 4),
    CS_VT3(SHAPE3_BOX, 4, 3, 16, 1, 4),  CS_VT3(SHAPE3_BOX, 4, 2, 16, 1, 4),
    CS_VT3(SHAPE3_BOX, 3, 3, 16, 1, 4),  CS_VT3(SHAPE3_BOX, 3, 2, 16, 1, 4),
    CS_VT3(SHAPE3_BOX, 2, 3, 16, 1, 4),  CS_VT3(SHAPE3_BOX, 2, 2, 16, 1, 4),
    CS_VT3(SHAPE3_BOX, 3, 3, 8, 1, 4),   CS_VT3(SHAPE3_BOX, 3, 2, 8, 1, 4),
    CS_VT3(SHAPE3_STAR, 8, 4, 8, 1, 2),  CS_VT3(SHAPE3_STAR, 8, 3, 8, 1, 2),  CS_VT3(SHAPE3_STAR, 8, 2, 8, 1, 2),
    CS_VT3(SHAPE3_STAR, 6, 4, 8, 1, 2),  CS_VT3(SHAPE3_STAR, 6, 3, 8, 1, 2),  CS_VT3(SHAPE3_STAR, 6, 2, 8, 1, 2),
    CS_VT3(SHAPE3_STAR, 3, 4, 16, 1, 4), CS_VT3(SHAPE3_STAR, 3, 3, 16, 1, 4), CS_VT3(SHAPE3_STAR, 3, 2, 16, 1, 4),
    CS_VT3(SHAPE3_STAR, 2, 4, 16, 1, 4), CS_VT3(SHAPE3_STAR, 2, 3, 16, 1, 4), CS_VT3(SHAPE3_STAR, 2, 2, 16, 1, 4),
    CS_VT3(SHAPE3_STAR, 3, 4, 8, 1, 4),  CS_VT3(SHAPE3_STAR, 3, 3, 8, 1, 4),  CS_VT3(SHAPE3_STAR, 3, 2, 8, 1, 4),
};

// Predicted us per step: a launch, plus the larger of its iterations (p + q kf us each; where two
// workgroups share a CU `two` times that) and its bytes (a read of every tile with its overlap, a write of
// the grid).  Fitted to 48-step runs of every variant on 17 grids from 64^3 to 512^3, flat and long
// ones among them: 5% (box) and 6% (star) rms; its choice took at most 1.03 times the fastest
// variant's time, once 1.14 (star, 150 x 300 x 300).
double tile3_cost(const Variant &v, int64_t nz, int64_t ny, int64_t nx) {
  struct Fit {
    int by, nw;
    double p, q;
  };
  static const Fit box[] = {{32, 16, 0.47, 0.518}, {24, 8, 0.48, 0.38},  {48, 16, 0.53, 0.76},
                            {64, 16, 0.68, 0.993}, {80, 16, 0.76, 1.28}, {64, 8, 1.22, 0.877}};
  static const Fit star[] = {{32, 16, 0.82, 0.126}, {24, 8, 0.59, 0.121}, {48, 16, 0.96, 0.198},
                             {48, 8, 0.74, 0.262},  {64, 8, 0.89, 0.356}};
  const bool b = v.shape == SHAPE3_BOX;
  const int wpe = v.by / v.nw >= 6 ? 2 : 4, slots = slots_of(v.nw, wpe);
  const Tile3Split sp = tile3_split(nz, ny, nx, v.by, v.kf, slots);
  const int64_t wgs = (int64_t)sp.tx * sp.ty * sp.zchunks, iters = (sp.zc + 3 * v.kf - 1 + 2) / 3 * 3;
  double it = 0.0;
  for (const Fit *f = b ? box : star, *e = f + (b ? 6 : 5); f < e; ++f)
    if (f->by == v.by && f->nw == v.nw) it = f->p + f->q * v.kf;
  if (slots > 256 && wgs > 256) it *= b ? 1.75 : 1.6;
  const double chain = (double)((wgs + slots - 1) / slots * iters) * it;
  const double bytes = 8.0 * ((double)wgs * 64 * v.by * (double)(sp.zc + 2 * v.kf) + (double)nz * ny * nx);
  return ((b ? 2.7 : 2.1) + std::max(chain, bytes / (b ? 4.47e6 : 5.23e6))) / v.kf;
}

const Variant *variants_3d_tile(int *count) {
  *count = (int)(sizeof(kVariantsTile3D) / sizeof(kVariantsTile3D[0]));
  return kVariantsTile3D;
}

}  // namespace cs
