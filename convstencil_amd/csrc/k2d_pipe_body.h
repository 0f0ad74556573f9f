// k2d_pipe_body.h -- level-pipelined register-streaming FP64 2-D kernels for gfx950.
//
// Replaces kernel2d (reference src/2d/gpu.cu:30-70) and its time loop (src/2d/gpu.cu:316-329,
// 336-425) on grids at least 512 columns wide.  The register-streaming kernels of k2d_reg.hip
// advance a strip of 64 PX columns KF steps inside one wave, so the partial sums of KF levels
// share one wave's registers: 4 columns per lane at depth 8 (radius 1), 2 at depth 4 (radius-3
// star), and the radius-3 box does not fit at all.  Narrow strips cost recomputed columns
// (2 R KF of 64 PX) and lane shifts (4 R moves per PX cells and level).  Here the levels of a
// strip are dealt over the NWV waves of a workgroup: wave w advances every row by levels
// w KFW .. w KFW + KFW - 1 and hands it to wave w + 1 through LDS.  A wave then holds KFW
// levels of 8 columns per lane: 512-column strips at 12 (box radius 1), 16 (star radius 1), 8
// (star radius 3) or 4 (box radius 3) steps per launch.
//
// What bounds them (profiles/fp64_pipe_tile_counters.md): the boxes FP64 issue and the power it draws.
// Vector instructions take 81% (radius 1) and 83% (radius 3) of the cycles, 91% and 96% of them are FMAs
// and multiplications, and the clock falls to 1.7-1.95 GHz on random data against 2.36 GHz on zeros, where the
// same cycles take 0.45 instead of 0.57 ms (10240^2, depth 12); so what is left to gain is work not done: recomputed
// rows and columns (11%).  The radius-3 star issues in 61% of the cycles (2.0 GHz): its one workgroup of eight waves
// per CU meets at a barrier every two rows with no other one to fill the waits.  HBM carries 2.1-3.2 TB/s.
// Measured, GStencil/s of the kernel alone, k2d_reg / k2d_f64 before and this kernel: box2d1r 10240^2 2037 ->
// 2280, star2d1r 10240^2 2140 -> 3440, star2d3r 8192^2 1013 -> 1208, box2d3r 8192^2 306 -> 458.
//
// Rows.  A wave's level s keeps partial sums for the 2R + 1 rows that the incoming row
// contributes to, as in k2d_reg.hip; the sum order per output is the same (rows dy = -R .. R,
// columns dx = -R .. R, one chain of FMAs), so results agree bit for bit.
//
// Hand-over.  A ring of S = 2 B row slots per pair of waves; a workgroup barrier closes every
// block of B rows (the last block of a barrier pattern of NSB rows may be shorter), wave w + 1
// reads the row that wave w wrote B rows ago, and a slot is written again B rows after it was
// read: both fall into another block.  Two workgroups per CU fill each other's waits (box
// radius 1 without any barrier: 2720 against 2690 GStencil/s without memory traffic).  A slot
// holds pair i of all lanes side by side (lane l: columns l PX + 2 i, + 1): 16-byte accesses at
// consecutive addresses, no bank conflicts, and the reader is the same lane.
//
// Memory.  The first wave loads and the last wave stores whole rows in memory order, 1 KiB
// per instruction, and turns them into each lane's run of PX columns through a staging row in
// LDS whose 16-byte pieces are rotated within groups of PX / 2 (piece p of every 64 at p with
// its low bits advanced by p / 16), which spreads both the linear and the by-lane accesses over
// all banks.  Straight from the lanes' runs each instruction touches 64 separate 64-byte
// segments: 0.85 against 0.73 ms per launch (depth 16, one box).
//
// Halo.  Strips start at column 0 and the last ends at column nx - 1 (neighbours overlap by at
// least 2 H columns; where the last two overlap further both store the same bits), so a
// halo column is only ever a lane shift's missing source: lane 0 or 63 of an outer strip.  If
// every halo cell that a workgroup's cells depend on is +0 in both buffers -- it looks once, at
// its start -- the shift's zero fill is the halo and outer strips run the inner strips' code
// (edge workgroups take the same time, 446 against 448 us); rows outside the interior are
// zeroed as they complete, in the blocks that hold such rows only.  Else the general form: the
// first wave loads the halo columns of both buffers beside each row with the row and keeps those
// of the last 64 rows in LDS, from where every level fills its shifts (loaded by every level for
// itself, a miss per row and level, edge workgroups took twice the time of inner ones); a halo row
// is loaded when a level needs it.  Level s takes its halo from the buffer that step s of the
// ping-pong would read (in, out, in, ...; Geo::flip exchanges them), which is exact for halos that
// differ between the buffers too.
//
// Priorities.  Of two waves on a SIMD the older one issues first, ends early (338 of 577 us)
// and leaves the other alone with its waits.  A wave lowers its priority at 50, 75 and 90% of
// its rows, so the one behind catches up: box2d1r 2210 -> 2290, box2d3r 445 -> 458.
#pragma once
#include <atomic>

#include "cs_internal.h"

namespace cs {

namespace {

typedef const double __attribute__((address_space(4))) cdouble;  // scalar loads
typedef const double __attribute__((address_space(1))) gdouble;
typedef double pair_t __attribute__((ext_vector_type(2)));

// One launch: strips of 64 PX columns x chunks of `rows` rows, one workgroup each.
struct PipeSplit {
  int strips, chunks;
  int64_t rows;
};

constexpr int modn(int v, int m) { return ((v % m) + m) % m; }

template <int R, int PX, int KFW, int NWV, int B>
struct Pipe2D {
  static constexpr int KF = KFW * NWV;
  static constexpr int H = R * KF;  // recomputed columns per side; warm-up rows
  static constexpr int W = 64 * PX;
  static constexpr int OX = W - 2 * H;
  static constexpr int NS = 2 * R + 1;  // partial-sum rows per level
  static constexpr int PP = PX / 2;     // 16-byte pieces per lane and row
  static constexpr int S = 2 * B;
  static constexpr int SKEW = B + R * KFW;  // rows a wave's input is behind that of the wave before it
  static constexpr int HR = 64;  // rows of the ring of halo columns (general form)
  // doubles: hand-overs, two staging rows for loads and stores, the halo columns of HR rows
  static constexpr int LDS = ((NWV - 1) * S + 4) * W + HR * 4 * R;
  static_assert((NWV - 1) * SKEW + R * KFW + 2 * B < HR, "the last wave reads halo columns of rows long past");
  static_assert(OX > 0 && NWV >= 2 && R <= PX, "strip too narrow");
  static_assert(H % 2 == 0, "outputs are stored in pairs of columns");
  static_assert(PP == 1 || PP == 2 || PP == 4, "staging rotates within groups of PP pieces");
};

// lane l gets lane l - 1's (lane_from_lower) or lane l + 1's value, the lane without a source f.
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

// A wave-uniform address, opaque to the compiler: it would otherwise compute every phase's
// halo addresses ahead of the loop and spill them.
__device__ __forceinline__ uint64_t opaque(const double *p) {
  const uint64_t v = (uint64_t)p;
  uint64_t u = (uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)v) |
               ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32);
  asm volatile("" : "+s"(u));
  return u;
}

enum { FIRST = 0, MID = 1, LAST = 2 };

// One wave's levels.  GEN: the general halo form.
template <int R, int SH, int PX, int KFW, int NWV, int B, int NSB, int RING, int ROLE, bool GEN>
struct Stage2D {
  using C = Pipe2D<R, PX, KFW, NWV, B>;
  static constexpr int D = 2 * R + 1, NS = C::NS, PP = C::PP, S = C::S, W2 = C::W / 2;
  static constexpr bool BOX = SH == SHAPE_BOX;
  // 49 weights do not fit the scalar registers: they are loaded again for every row of taps
  static constexpr bool WLOAD = BOX && R > 1;
  static constexpr int PER = ROLE == FIRST ? reg_period((NSB - 1) / 2, RING) : NSB;
  static_assert(NSB % NS == 0 && NSB % 2 == 1, "barrier pattern");

  const double *in;
  double *out;
  const double *wts;
  double w[WLOAD ? 1 : D * D];
  pair_t *from, *to;   // hand-over rings (this lane's piece 0 of slot 0)
  pair_t *stage;       // two staging rows
  int pos[PP];         // where this lane's pieces lie in a staging row
  unsigned load_off;   // FIRST: byte offset of this lane's piece of a row's first KiB
  int store_off[PP];   // LAST: byte offsets in a row of the pieces this lane stores
  int64_t ny, nx, pitch, ey, oy, ox, xs;
  int par;  // whether level 0 of this wave takes its halo from `in` (0) or `out` (1)
  int lane;
  pair_t raw[ROLE == FIRST ? RING : 1][PP];  // rows in flight
  // general form: a ring of the halo columns beside HR rows, [row][buffer][left R, right R]; lane
  // l < 4 R of the first wave loads the l-th entry of every row, with the row
  double *side;
  const double *side_src;
  double side_raw[ROLE == FIRST && GEN ? RING : 1];
  double acc[KFW][NS][PX];

  // Selects between copies of the two pointers: selecting between the members themselves takes their
  // addresses, and the whole Stage2D, partial sums included, then lives in scratch memory (40 steps
  // with an uploaded halo: box radius 1 3000^2 1624 -> 321 us, star radius 3 6000^2 3642 -> 1507).
  __device__ __forceinline__ const double *halo_buffer(int s) const {
    const double *const a = in, *const b = out;
    return ((par + s) & 1) ? b : a;
  }
  __device__ __forceinline__ int64_t clamped(int64_t y) const {
    const int64_t ay = oy + y;
    return ay < 0 ? 0 : ay >= ey ? ey - 1 : ay;
  }

  // Row r in memory order, the row clamped into the array: a row outside it lies more than R
  // rows from the interior and reaches no output.
  __device__ __forceinline__ void load_row(int64_t r, pair_t (&dst)[PP], double &h) {
    const int64_t ay = clamped(r);
    const char *p = (const char *)(in + ay * pitch + ox + xs) + load_off;
    if constexpr (ROLE == FIRST && GEN) h = side_src[ay * pitch];
#pragma unroll
    for (int i = 0; i < PP; ++i) {
      dst[i].x = *(const double *)(p + i * 1024);
      dst[i].y = *(const double *)(p + i * 1024 + 8);
    }
  }

  __device__ __forceinline__ void stage_row(int64_t r, pair_t *st, const pair_t (&v)[PP], double h) {
#pragma unroll
    for (int i = 0; i < PP; ++i) st[i * 64 + lane] = v[i];
    if constexpr (ROLE == FIRST && GEN) {
      if (lane < 4 * R) side[((int)r & (C::HR - 1)) * 4 * R + lane] = h;
    }
  }

  // qe[R + c] = cell c of the lane's run in row y of level s, c = -R .. PX + R - 1
  __device__ __forceinline__ void extend(const double (&q)[PX], double (&qe)[PX + 2 * R], int64_t y, int s) {
#pragma unroll
    for (int j = 0; j < PX; ++j) qe[R + j] = q[j];
    if constexpr (GEN) {
      const double *h = side + ((int)y & (C::HR - 1)) * 4 * R + ((par + s) & 1) * 2 * R;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        qe[k] = lower_or(q[PX - R + k], h[k]);
        qe[PX + R + k] = upper_or(q[k], h[R + k]);
      }
    } else {
#pragma unroll
      for (int k = 0; k < R; ++k) {
        qe[k] = lane_from_lower(q[PX - R + k]);
        qe[PX + R + k] = lane_from_upper(q[k]);
      }
    }
  }

  // A row outside the interior is its level's halo, not what the taps made of it.
  __device__ __forceinline__ void halo_row(double (&q)[PX], int64_t y, int s) {
    if (y >= 0 && y < ny) return;  // wave-uniform
    if constexpr (GEN) {
      gdouble *p = (gdouble *)opaque(halo_buffer(s) + clamped(y) * pitch + ox + xs);
#pragma unroll
      for (int j = 0; j < PX; ++j) q[j] = p[lane * PX + j];
    } else {
#pragma unroll
      for (int j = 0; j < PX; ++j) q[j] = 0.0;
    }
  }

  // Phase `it + K`: this wave's input row ys + it + K through its KFW levels.  CHK: the
  // block holds rows outside the interior.
  template <int K, bool CHK>
  __device__ __forceinline__ void phase(int64_t it, int64_t ys, int64_t y0, int64_t y1, int &slot) {
    const int64_t r = ys + it + K;
    double q[PX];
    pair_t done[PP];
    if constexpr (ROLE == FIRST) {
      // row r was staged in the phase before; row r + 1 has arrived and is staged now
      pair_t *st = stage + ((it + K) & 1) * W2, *next = stage + ((it + K + 1) & 1) * W2;
#pragma unroll
      for (int j = 0; j < PP; ++j) {
        const pair_t v = st[pos[j]];
        q[2 * j] = v.x;
        q[2 * j + 1] = v.y;
      }
      constexpr int N = (K + 1) % RING, NH = GEN ? N : 0;
      stage_row(r + 1, next, raw[N], side_raw[NH]);
      load_row(r + 1 + RING, raw[N], side_raw[NH]);
      // loaded from `in`; with Geo::flip the halo rows of level 0 are those of `out`
      if constexpr (GEN && CHK) halo_row(q, r, 0);
    } else {
      const pair_t *p = from + (slot >= B ? slot - B : slot - B + S) * W2;
#pragma unroll
      for (int j = 0; j < PP; ++j) {
        const pair_t v = p[j * 64];
        q[2 * j] = v.x;
        q[2 * j + 1] = v.y;
      }
    }
    if constexpr (ROLE == LAST) {
      // the output row staged in the phase before, in memory order
      const pair_t *st = stage + ((it + K + 1) & 1) * W2;
#pragma unroll
      for (int i = 0; i < PP; ++i) done[i] = st[i * 64 + lane];
    }
#pragma unroll
    for (int s = 0; s < KFW; ++s) {
      const int64_t yq = r - R * s;
      double qe[PX + 2 * R];
      extend(q, qe, yq, s);
#pragma unroll
      for (int dy = R; dy >= -R; --dy) {
        // the taps of row offset dy into row yq - dy (dy = R completes it, dy = -R starts it)
        double(&T)[PX] = acc[s][modn(K - R * s - dy, NS)];
        double wr[D], t[PX];
        if constexpr (WLOAD) {
          cdouble *p = (cdouble *)opaque(wts) + (dy + R) * D;
#pragma unroll
          for (int i = 0; i < D; ++i) wr[i] = p[i];
        } else {
#pragma unroll
          for (int i = 0; i < D; ++i) wr[i] = w[(dy + R) * D + i];
        }
#pragma unroll
        for (int dx = -R; dx <= R; ++dx) {
          if (!BOX && dy != 0 && dx != 0) continue;
          const bool start = BOX || dy == 0 ? dx == -R : dx == 0;  // the row's first tap
#pragma unroll
          for (int j = 0; j < PX; ++j) {
            const double v = qe[R + j + dx];
            t[j] = start && dy == -R ? wr[dx + R] * v : __builtin_fma(wr[dx + R], v, start ? T[j] : t[j]);
          }
        }
#pragma unroll
        for (int j = 0; j < PX; ++j) T[j] = t[j];
        // keep the partial sums computed here (see k2d_reg.hip)
        if (dy < R) {
#pragma unroll
          for (int j = 0; j < PX; ++j) asm volatile("" : "+v"(T[j]));
        }
      }
      const double(&A)[PX] = acc[s][modn(K - R * s - R, NS)];
#pragma unroll
      for (int j = 0; j < PX; ++j) q[j] = A[j];
      if constexpr (CHK) {
        if (ROLE != LAST || s + 1 < KFW) halo_row(q, yq - R, s + 1);  // the last level's row is an output
      }
      if constexpr (ROLE == LAST) {
        if (s == 0) {
          // a row outside [y0, y1) gets an empty range: every phase issues the same stores
          const int64_t yo = r - 1 - R * KFW;
          const bool ok = yo >= y0 && yo < y1;
          const __amdgpu_buffer_rsrc_t rs = buffer_over(out + (oy + yo) * pitch + ox + xs, ok ? C::W * 8 : 0);
#pragma unroll
          for (int i = 0; i < PP; ++i) buffer_store2(rs, store_off[i], done[i].x, done[i].y);
        }
      }
    }
    if constexpr (ROLE == LAST) {
      pair_t *st = stage + ((it + K) & 1) * W2;
#pragma unroll
      for (int j = 0; j < PP; ++j) {
        pair_t v;
        v.x = q[2 * j];
        v.y = q[2 * j + 1];
        st[pos[j]] = v;
      }
    } else {
      pair_t *p = to + slot * W2;
#pragma unroll
      for (int j = 0; j < PP; ++j) {
        pair_t v;
        v.x = q[2 * j];
        v.y = q[2 * j + 1];
        p[j * 64] = v;
      }
    }
    slot = slot + 1 == S ? 0 : slot + 1;
    // the same pattern in every wave of the workgroup: all run the same number of phases
    if constexpr ((K % NSB) % B == B - 1 || K % NSB == NSB - 1) lds_barrier();
  }

  template <int K, bool CHK>
  __device__ __forceinline__ void phases(int64_t it, int64_t ys, int64_t y0, int64_t y1, int &slot) {
    if constexpr (K < PER) {
      phase<K, CHK>(it, ys, y0, y1, slot);
      phases<K + 1, CHK>(it, ys, y0, y1, slot);
    }
  }

  // `iters` phases (a multiple of every role's period) from input row ys on.
  __device__ __forceinline__ void run(int64_t ys, int64_t y0, int64_t y1, int64_t iters) {
#pragma unroll
    for (int s = 0; s < KFW; ++s)
#pragma unroll
      for (int k = 0; k < NS; ++k)
#pragma unroll
        for (int j = 0; j < PX; ++j) acc[s][k][j] = 0.0;
    if constexpr (ROLE == FIRST) {
      load_row(ys, raw[0], side_raw[0]);
      stage_row(ys, stage, raw[0], side_raw[0]);
#pragma unroll
      for (int k = 1; k <= RING; ++k) {
        load_row(ys + k, raw[k % RING], side_raw[GEN ? k % RING : 0]);
        __builtin_amdgcn_sched_barrier(0);  // in order, so that the first wait is not for the youngest
      }
    }
    int slot = 0;
    int64_t it = 0;
    // three loops, not one with a branch: the branch's copies of the partial sums spilled
    for (; it < iters && ys + it < R * KFW; it += PER) phases<0, true>(it, ys, y0, y1, slot);
    // a block without checks ends before the first row that completes outside the interior (in
    // the first wave's general form: that enters outside it)
    const int64_t end = ny + (ROLE == FIRST && GEN ? 0 : R) - PER + 1 - ys;
    const int64_t inner = end < iters ? end : iters;
    const int64_t t1 = iters / 2, t2 = iters * 3 / 4, t3 = iters * 9 / 10;
    __builtin_amdgcn_s_setprio(3);
    for (; it < inner; it += PER) {
      if (it >= t1 && it < t1 + PER) __builtin_amdgcn_s_setprio(2);
      if (it >= t2 && it < t2 + PER) __builtin_amdgcn_s_setprio(1);
      if (it >= t3 && it < t3 + PER) __builtin_amdgcn_s_setprio(0);
      phases<0, false>(it, ys, y0, y1, slot);
    }
    for (; it < iters; it += PER) phases<0, true>(it, ys, y0, y1, slot);
  }
};

template <int R, int SH, int PX, int KFW, int NWV, int B, int NSB, int RING, int ROLE, bool GEN>
__device__ __forceinline__ void run_stage(const double *in, double *out, const double *wts, const Geo &g, int64_t xs,
                                          bool left, bool right, int64_t y0, int64_t y1, int lane, int wv,
                                          double *lds) {
  using C = Pipe2D<R, PX, KFW, NWV, B>;
  using T = Stage2D<R, SH, PX, KFW, NWV, B, NSB, RING, ROLE, GEN>;
  T t;
  t.in = in;
  t.out = out;
  t.wts = wts;
  if constexpr (!T::WLOAD) {
#pragma unroll
    for (int i = 0; i < T::D * T::D; ++i) t.w[i] = wts[i];
  }
  t.ny = g.n[1];
  t.nx = g.n[2];
  t.pitch = g.ext[2];
  t.ey = g.ext[1];
  t.oy = g.org[1];
  t.ox = g.org[2];
  t.xs = xs;
  t.lane = lane;
  t.par = (wv * KFW + (int)g.flip) & 1;
  pair_t *l2 = (pair_t *)lds;
  t.from = l2 + (wv - 1) * C::S * T::W2 + lane;
  t.to = l2 + wv * C::S * T::W2 + lane;
  t.stage = l2 + ((NWV - 1) * C::S + (ROLE == LAST ? 2 : 0)) * T::W2;
  t.side = lds + ((NWV - 1) * C::S + 4) * C::W;
  if constexpr (ROLE == FIRST && GEN) {
    const int e = lane % (4 * R), k = e % (2 * R);
    t.side_src = (e < 2 * R ? in : (const double *)out) + t.ox + (k < R ? k - R : t.nx + k - R);
  }
#pragma unroll
  for (int j = 0; j < C::PP; ++j) {
    const int c = C::PP * lane + j, p = c & 63;  // piece c of the row, p of its KiB
    t.pos[j] = (c & ~63) + (p & ~(C::PP - 1)) + ((p + (p >> 4)) & (C::PP - 1));
    // the piece at position 64 j + lane, as a column
    const int col = 2 * (64 * j + (lane & ~(C::PP - 1)) + ((lane - (lane >> 4)) & (C::PP - 1)));
    if (j == 0) t.load_off = col * 8;
    const bool ok = (left || col >= C::H) && (right || col < C::W - C::H);
    t.store_off[j] = ok ? col * 8 : kBufferDrop;
  }
  constexpr int P = reg_period((NSB - 1) / 2, RING);  // FIRST's period, a multiple of the others'
  const int64_t need = (y1 - y0) + 2 * C::H + (NWV - 1) * B + 1;
  t.run(y0 - C::H - (int64_t)wv * C::SKEW, y0, y1, (need + P - 1) / P * P);
}

template <int R, int SH, int PX, int KFW, int NWV, int B, int NSB, int RING>
__global__ __launch_bounds__(NWV * 64, 2) void k2d_pipe(const double *in, double *out, const double *wts, Geo g,
                                                       PipeSplit sp) {
  using C = Pipe2D<R, PX, KFW, NWV, B>;
  extern __shared__ __attribute__((aligned(16))) double pipe_lds[];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chunk = __builtin_amdgcn_readfirstlane(blockIdx.x / (unsigned)sp.strips);
  const int strip = (int)blockIdx.x - chunk * sp.strips;
  const int64_t ny = g.n[1], nx = g.n[2], pitch = g.ext[2];
  const int64_t y0 = chunk * sp.rows, y1 = y0 + sp.rows < ny ? y0 + sp.rows : ny;
  const bool left = strip == 0, right = strip == sp.strips - 1;
  const int64_t xs = right ? nx - C::W : (int64_t)strip * C::OX;
  bool general = false;
  if (left || right || y0 < C::H || y1 + C::H > ny) {
    // any halo cell in reach that is not +0, in either buffer (rows -R .. ny + R - 1 beside
    // the strip, columns of the strip above and below)
    const int64_t ya = y0 - C::H < -R ? -R : y0 - C::H, yb = y1 + C::H > ny + R ? ny + R : y1 + C::H;
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
          if (ya < 0) any |= (uint64_t)__double_as_longlong(p[(k - R) * pitch + x]);
          if (yb > ny) any |= (uint64_t)__double_as_longlong(p[(ny + k) * pitch + x]);
        }
      }
    }
    general = __syncthreads_or(any != 0);
  }
#define CS_ROLE(ROLE)                                                                                              \
  do {                                                                                                             \
    if (general)                                                                                                   \
      run_stage<R, SH, PX, KFW, NWV, B, NSB, RING, ROLE, true>(in, out, wts, g, xs, left, right, y0, y1, lane, wv, \
                                                               pipe_lds);                                          \
    else                                                                                                           \
      run_stage<R, SH, PX, KFW, NWV, B, NSB, RING, ROLE, false>(in, out, wts, g, xs, left, right, y0, y1, lane,    \
                                                                wv, pipe_lds);                                     \
  } while (0)
  if (wv == 0) {
    CS_ROLE(FIRST);
  } else if (wv == NWV - 1) {
    CS_ROLE(LAST);
  } else if constexpr (NWV > 2) {
    CS_ROLE(MID);
  }
#undef CS_ROLE
}

template <int R, int SH, int PX, int KFW, int NWV, int B, int NSB, int RING>
struct PipeVariant {
  using C = Pipe2D<R, PX, KFW, NWV, B>;
  static constexpr size_t kLds = C::LDS * sizeof(double);
  // resident workgroups on each device, 0 where prepare() has not run: the LDS attribute belongs to
  // one device's copy of the kernel
  static constexpr int kDevices = 64;
  static std::atomic<int64_t> slots[kDevices];

  static hipError_t prepare() {
    int nb = 0, dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const bool known = dev >= 0 && dev < kDevices;
    if (known && slots[dev].load(std::memory_order_relaxed) > 0) return hipSuccess;
    const void *f = (const void *)k2d_pipe<R, SH, PX, KFW, NWV, B, NSB, RING>;
    if ((e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds)) != hipSuccess) return e;
    if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, NWV * 64, kLds)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    if (known) slots[dev].store((int64_t)(nb > 0 ? nb : 1) * (cus > 0 ? cus : 1), std::memory_order_relaxed);
    return hipSuccess;
  }

  static hipError_t launch(const double *in, double *out, const double *wts, const Geo &g, hipStream_t s) {
    int dev = 0;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const int64_t ny = g.n[1], nx = g.n[2];
    const int64_t n = dev >= 0 && dev < kDevices ? slots[dev].load(std::memory_order_relaxed) : 0;
    if (nx < C::W || ny < 1) return hipErrorInvalidValue;  // strips are 64 PX columns of the interior
    PipeSplit sp;
    const int64_t strips = 1 + (nx - C::W + C::OX - 1) / C::OX;
    int64_t chunks = (n > 0 ? n : 256) / strips;  // every workgroup resident at once
    if (chunks > ny) chunks = ny;
    if (chunks < 1) chunks = 1;
    sp.rows = (ny + chunks - 1) / chunks;
    chunks = (ny + sp.rows - 1) / sp.rows;
    if (strips * chunks > 0x7fffffff) return hipErrorInvalidValue;
    sp.strips = (int)strips;
    sp.chunks = (int)chunks;
    hipLaunchKernelGGL((k2d_pipe<R, SH, PX, KFW, NWV, B, NSB, RING>), dim3((unsigned)(strips * chunks)),
                       dim3(NWV * 64), kLds, s, in, out, wts, g, sp);
    return hipGetLastError();
  }
};

template <int R, int SH, int PX, int KFW, int NWV, int B, int NSB, int RING>
std::atomic<int64_t> PipeVariant<R, SH, PX, KFW, NWV, B, NSB, RING>::slots[kDevices] = {};

}  // namespace

// Variant::mf 10 marks this family: by = 1 (rows are chunked per launch), bx = output columns
// per workgroup, px = columns per lane, st = rows in flight in the first wave; the weights are
// the dense (2R+1)^2 block.
#define CS_VP2D(ID, R, SH, PX, KFW, NWV, B, RING)                                                           \
  Variant {                                                                                                 \
    ID, 10, R, SH, KFW *NWV, 1, Pipe2D<R, PX, KFW, NWV, B>::OX, NWV,                                        \
        PipeVariant<R, SH, PX, KFW, NWV, B, 2 * R + 1, RING>::kLds, PX, RING,                               \
        &PipeVariant<R, SH, PX, KFW, NWV, B, 2 * R + 1, RING>::launch,                                      \
        &PipeVariant<R, SH, PX, KFW, NWV, B, 2 * R + 1, RING>::prepare,                                     \
        "k2d_pipe<r" #R "," #SH ",p" #PX "," #KFW "x" #NWV ",b" #B ",ring" #RING ">"                        \
  }


}  // namespace cs
