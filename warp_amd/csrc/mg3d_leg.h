// One leg of the V-cycle on a coarse level in one launch.  Included by
// mg3d.hip.
//
// On a coarse level each step of vcycle (f3d_mgrid.F:1101-1591) -- a half
// sweep, its boundary conditions, the residual and its conductor records,
// the restriction, the expansion -- is a launch of 4-10 us that moves little:
// its time is the launch, the first loads after it and the z-march's serial
// chain.  Here a block takes a tile of the level with the halo that the leg's
// steps need, brings it to LDS once and runs every step there, each on a
// region one point smaller than the step before, so that nothing passes
// between blocks:
//   k_leg_down: phi = 0, half sweep 0, half sweep 1, residual, restriction;
//   k_leg_up:   expansion from the coarser level, half sweeps 0 and 1.
// The up leg writes the level's second phi buffer (blocks beside it still read
// the first), which is where the finer level's expansion then reads it.
//
// Each point is evaluated with the expressions of the kernels that these
// replace, in the same order, so the results are the same bits, however often
// a halo point is computed.  The boundary conditions become rules for
// addresses: at a Neumann face the neighbour beyond is the one before it, in a
// periodic axis coordinates run on and are wrapped when memory is read, and
// Dirichlet faces hold zero (the error's value there).
//
// Measured (launch time in a replayed V-cycle, FP64): 32x32x64 nodes without
// conductors 10.9 us down and 9.3 us up, where three launches each took 13
// and 16 us; 64x64x128 with the pipe and the annulus 20.7 and 26.9 us against
// 31 and 26 us, 32x32x64 14.1 and 11.4 against 22 and 19.  A solve of
// 128x128x256 with them 2.45 -> 2.16 ms, of 101x75x190 with Neumann faces
// 3.50 -> 2.16 ms (~600 boundary launches of 3-5 us less).
#pragma once
#include "mg3d_kernels.h"

// Such a kernel is a chain of latencies (a memory round trip is 1 us, an LDS
// round trip with the sum behind it 0.2 us), so everything a block reads is
// asked for at its start: the tile's numbers from one table, rho and the
// points' classes (and phi) with all of a thread's loads in flight, the
// transfer tables, the records' constants into registers.  A thread owns the
// same pairs of neighbouring points in every step, whose coordinates it
// decodes once into a word per point.
// What a block reads about its tile along one axis.
struct LegTile {
  int r0, r1;      // down: the residual's range; up: the fine nodes it writes
  int own0, own1;  // the fine nodes whose phi the tile writes
  int c0, c1;      // coarse nodes (up: coarse window, running on over a periodic face)
  int pad0, pad1;
};

// One axis of a level and of its tiles.
struct LegAxis {
  int n, bm, bp;       // cells, boundary types
  int nt, ts;          // tiles, and coarse (down) or fine (up) nodes per tile
  int ext;             // window points, the largest of all tiles
  int nc, cmin, cmax;  // coarse cells, computed coarse range
  const int *lo, *hi;  // restriction windows and weights (5 per coarse node)
  const double *rw;
  const int *ej;       // expansion: coarse index and weight per fine node
  const double *ew;
  int cext;            // (up) coarse window points
  const LegTile *tile;
};

// A conductor record of a tile's window: local coordinates (8 bits each) with
// the sides of LEGP_RAW (6 bits), and (colour << 31) | index.
struct LegRec {
  uint32_t at, rec;
};

template <typename T>
struct LegArgs {
  RBGeom g, gc;
  LegAxis a[3];
  uint32_t mhx, my, mcx, mcy;      // reciprocals of the decoding divisors
  int plain;                       // windows of three in a row everywhere (restriction)
  int mirror;                      // a Neumann face somewhere
  int ni;                          // pairs per thread
  T sx, sy, sz, spm1;              // half sweep
  T rx, ry, rz, mgparam;           // residual
  double ff;
  const uint8_t *cls;              // class per element and the sides of LEGP_RAW << 2 (NULL: all dense)
  const uint32_t *first;           // a tile's records: rec[first[t]] .. rec[first[t+1]]
  const LegRec *rec;               // NULL: none
  SubList<T> sor[2], res[2];
};

enum { LEG_DENSE = 0, LEG_REC = 1, LEG_INT = 2 };
constexpr int LEG_TH = 512;  // threads of a block
constexpr int LEG_NI = 4;    // pairs of points per thread, at most
// Coarse nodes of a tile along one axis, at most (down); points of a window.
constexpr int LEG_CMAX = 16, LEG_WMAX = 32;

__device__ inline int leg_div(int t, uint32_t m) { return (int)__umulhi((uint32_t)t, m); }

// One axis of a tile: its window [w0, w1], the regions of the steps, in
// coordinates that run on over a periodic face.
struct LegWin {
  int w0, w1;
};

__device__ inline LegWin leg_clip(const LegAxis &a, int lo, int hi) {
  return a.bm == 2 ? LegWin{lo, hi} : LegWin{max(lo, 0), min(hi, a.n)};
}

__device__ inline int leg_wrap(const LegAxis &a, int i) {
  if (a.bm != 2) return i;
  return i < 0 ? i + a.n : i >= a.n ? i - a.n : i;
}

__device__ inline bool leg_swept(const LegAxis &a, int i) {
  return a.bm == 2 || ((i > 0 || a.bm != 0) && (i < a.n || a.bp != 0));
}

// LDS strides of the neighbours of a point (mirrored at Neumann faces).
struct LegNb {
  int xm, xp, ym, yp, zm, zp;
};

// A point's word: the steps it takes part in (0-3: the steps' regions lie one
// inside the other), the faces it mirrors at, whether the tile writes it,
// interior conductor point, record, the sides across which it reads an
// interior point before its pin.
enum {
  LEGP_DEPTH = 3,
  LEGP_MIRROR = 4,
  LEGP_OWN = 256,
  LEGP_INT = 512,
  LEGP_REC = 1024,
  LEGP_RAW = 2048
};

// raw (not 0): the first half sweep after the expansion.  The reference fills
// the guard points before it pins, so a point on a face reads an interior
// neighbour across it as it was before the pin; that value stands raw elements
// behind the point, in the place of its rho.
__device__ inline LegNb leg_nb(uint32_t p, int ex, int sz, int raw) {
  LegNb q{-1, 1, -ex, ex, -sz, sz};
  if (p & (63u * LEGP_MIRROR)) {
    if (p & (LEGP_MIRROR << 0)) q.xm = 1;
    if (p & (LEGP_MIRROR << 1)) q.xp = -1;
    if (p & (LEGP_MIRROR << 2)) q.ym = ex;
    if (p & (LEGP_MIRROR << 3)) q.yp = -ex;
    if (p & (LEGP_MIRROR << 4)) q.zm = sz;
    if (p & (LEGP_MIRROR << 5)) q.zp = -sz;
  }
  if (raw && (p & (63u * LEGP_RAW))) {
    if (p & (LEGP_RAW << 0)) q.xm += raw;
    if (p & (LEGP_RAW << 1)) q.xp += raw;
    if (p & (LEGP_RAW << 2)) q.ym += raw;
    if (p & (LEGP_RAW << 3)) q.yp += raw;
    if (p & (LEGP_RAW << 4)) q.zm += raw;
    if (p & (LEGP_RAW << 5)) q.zp += raw;
  }
  return q;
}

template <typename T>
__device__ inline uint32_t leg_mirror(const LegArgs<T> &A, int x, int y, int z) {
  if (!A.mirror) return 0u;
  uint32_t p = 0;
  const LegAxis &X = A.a[0], &Y = A.a[1], &Z = A.a[2];
  if (x == 0 && X.bm == 1) p |= LEGP_MIRROR << 0;
  if (x == X.n && X.bp == 1) p |= LEGP_MIRROR << 1;
  if (y == 0 && Y.bm == 1) p |= LEGP_MIRROR << 2;
  if (y == Y.n && Y.bp == 1) p |= LEGP_MIRROR << 3;
  if (z == 0 && Z.bm == 1) p |= LEGP_MIRROR << 4;
  if (z == Z.n && Z.bp == 1) p |= LEGP_MIRROR << 5;
  return p;
}

__device__ inline bool leg_in(const LegWin *r, int x, int y, int z) {
  return x >= r[0].w0 && x <= r[0].w1 && y >= r[1].w0 && y <= r[1].w1 && z >= r[2].w0 &&
         z <= r[2].w1;
}

// How many of an axis' nested regions hold coordinate i (bits 0-1), and
// whether the tile writes it (bit 2).
__device__ inline uint32_t leg_depth(const LegWin &r0, const LegWin &r1, const LegWin &r2,
                                     const LegWin &own, int i) {
  auto in = [&](const LegWin &r) { return (uint32_t)(i - r.w0) <= (uint32_t)(r.w1 - r.w0); };
  return (in(r0) ? 1u : 0u) + (in(r1) ? 1u : 0u) + (in(r2) ? 1u : 0u) + (in(own) ? 4u : 0u);
}

// A thread's pairs: the words of the two points by colour, the LDS element of
// the pair's first point, and which of the two has colour 0.
struct LegPts {
  uint32_t w[LEG_NI][2];
  int e[LEG_NI];
  uint32_t odd, single;  // single: the row ends with the pair's first point
  __device__ bool last(int i) const { return (single >> i) & 1u; }
};

// rho, the classes and (UP) phi of the window [r0] to LDS, and the thread's
// words for the nested regions r0, r1, r2.
template <typename T, bool UP>
__device__ inline void leg_load(const LegArgs<T> &A, const LegWin *r0, const LegWin *r1,
                                const LegWin *r2, const LegWin *own, const T *__restrict__ rho,
                                const T *__restrict__ phi, T *ph, T *rh, LegPts &P) {
  const int ex = A.a[0].ext, ey = A.a[1].ext, ez = A.a[2].ext, hx = (ex + 1) >> 1;
  const int items = hx * ey * ez;
  T v[LEG_NI][2], f[LEG_NI][2];
  uint8_t cl[LEG_NI][2];
  P.odd = P.single = 0;
#pragma unroll
  for (int i = 0; i < LEG_NI; i++) {
    P.e[i] = -1;
    P.w[i][0] = P.w[i][1] = 0;
    if (i >= A.ni) continue;
    const int t = threadIdx.x + i * LEG_TH;
    const int row = leg_div(t, A.mhx), h = t - row * hx;
    const int lz = leg_div(row, A.my), ly = row - lz * ey;
    const int x = r0[0].w0 + 2 * h, y = r0[1].w0 + ly, z = r0[2].w0 + lz;
    uint32_t dy = leg_depth(r0[1], r1[1], r2[1], own[1], y);
    uint32_t dz = leg_depth(r0[2], r1[2], r2[2], own[2], z);
    if (t < items) P.e[i] = 2 * h + ex * row;
    else dy = 0;
    const uint32_t own2 = dy & dz & 4u, d2 = min(dy & 3u, dz & 3u);
    const bool rowsw = leg_swept(A.a[1], y) && leg_swept(A.a[2], z);
    const int par = (x + y + z) & 1;
    P.odd |= (uint32_t)par << i;
    P.single |= (uint32_t)(2 * h + 1 >= ex) << i;
    const int py = leg_wrap(A.a[1], y), pz = leg_wrap(A.a[2], z);
    const int base = A.g.W * (py + 1 + A.g.PY * (pz + 1)), cs = (int)A.g.cs;
#pragma unroll
    for (int p = 0; p < 2; p++) {
      const uint32_t dx = leg_depth(r0[0], r1[0], r2[0], own[0], x + p);
      const bool sw = rowsw && leg_swept(A.a[0], x + p);
      uint32_t q = sw ? min(dx & 3u, d2) : 0u;
      const int px = leg_wrap(A.a[0], x + p);
      // points outside read the first element (unused)
      const int e = q ? base + ((px + 1) >> 1) + ((px + py + pz) & 1 ? cs : 0) : 0;
      v[i][p] = rho[e];
      f[i][p] = UP ? phi[e] : (T)0.;
      cl[i][p] = A.cls ? A.cls[e] : (uint8_t)LEG_DENSE;
      if (q && A.mirror) q |= leg_mirror(A, x + p, y, z);
      if (own2 & dx) q |= LEGP_OWN;
      P.w[i][p] = q;
    }
  }
#pragma unroll
  for (int i = 0; i < LEG_NI; i++) {
    if (i >= A.ni) continue;
#pragma unroll
    for (int p = 0; p < 2; p++) {
      uint32_t q = P.w[i][p];
      const bool sw = q & LEGP_DEPTH;
      // the conductor points take no part; interior ones where their phi or
      // residual is asked for
      const int cls = cl[i][p] & 3;
      if (UP && sw && cls == LEG_DENSE) q |= (uint32_t)(cl[i][p] >> 2) * LEGP_RAW;
      if (sw && cls != LEG_DENSE)
        q = (q & LEGP_OWN) | (cls == LEG_REC                ? LEGP_REC
                              : UP || (q & LEGP_DEPTH) == 3u ? LEGP_INT
                                                             : 0u);
      // (the second point of a row's last pair may be the next row's first)
      if (P.e[i] >= 0 && (p == 0 || !P.last(i))) {
        ph[P.e[i] + p] = sw ? f[i][p] : (T)0.;
        rh[P.e[i] + p] = sw ? v[i][p] : (T)0.;
      } else {
        q = 0;
      }
      P.w[i][p] = q;
    }
    if ((P.odd >> i) & 1u) {
      const uint32_t q = P.w[i][0];
      P.w[i][0] = P.w[i][1];
      P.w[i][1] = q;
    }
  }
}

// LDS element of a pair's point of colour c.
__device__ inline int leg_el(const LegPts &P, int i, int c) {
  return P.e[i] + (int)(((P.odd >> i) & 1u) ^ (uint32_t)c);
}

// A record's constants, for the half sweeps and (RES) the residual.
template <typename T, bool RES>
struct LegRecord {
  uint32_t at, rec, modes, rmodes;
  T k[6], denom, rk[6], rdenom, fac;
};

template <typename T, bool RES>
__device__ inline void leg_load_record(const LegArgs<T> &A, LegRec q, LegRecord<T, RES> &R) {
  const int c = (int)(q.rec >> 31), i = (int)(q.rec & 0x7fffffffu);
  R.at = q.at;
  R.rec = q.rec;
  const SubList<T> &s = c ? A.sor[1] : A.sor[0];
  R.modes = s.modes[i];
  R.denom = s.denom[i];
#pragma unroll
  for (int j = 0; j < 6; j++) R.k[j] = s.k[6 * i + j];
  if (RES) {
    const SubList<T> &r = c ? A.res[1] : A.res[0];
    R.rmodes = r.modes[i];
    R.rdenom = r.denom[i];
    R.fac = r.fac[i];
#pragma unroll
    for (int j = 0; j < 6; j++) R.rk[j] = r.k[6 * i + j];
  }
}

// The records of colour c inside r: half sweep (sor_record) or, with res, the
// residual (residual_record).  first: phi is zero everywhere, the
// neighbours, which may lie outside the window, are read from the point.  raw:
// leg_nb.
template <typename T, bool RES>
__device__ inline void leg_records(const LegArgs<T> &A, const LegWin *w, const LegWin *r, int c,
                                   bool res, bool first, int raw, T *ph, T *rh, int rec0, int nrec,
                                   const LegRecord<T, RES> &mine) {
  const int ex = A.a[0].ext, ey = A.a[1].ext, sz = ex * ey;
  // (the last threads first: they own the fewest pairs)
#pragma unroll 1
  for (int i = LEG_TH - 1 - (int)threadIdx.x; i < nrec; i += LEG_TH) {
    LegRecord<T, RES> R = mine;
    if (i >= LEG_TH) leg_load_record<T, RES>(A, A.rec[rec0 + i], R);
    const int lx = R.at & 255u, ly = (R.at >> 8) & 255u, lz = (R.at >> 16) & 255u;
    const int x = w[0].w0 + lx, y = w[1].w0 + ly, z = w[2].w0 + lz;
    if ((int)(R.rec >> 31) != c || !leg_in(r, x, y, z)) continue;
    const int e = lx + ex * (ly + ey * lz);
    LegNb q{0, 0, 0, 0, 0, 0};
    if (!first) q = leg_nb(leg_mirror(A, x, y, z) | (R.at >> 24) * LEGP_RAW, ex, sz, raw);
    uint32_t m = R.modes;
    T k[6];
#pragma unroll
    for (int j = 0; j < 6; j++) k[j] = R.k[j];
    if (RES && res) {
      m = R.rmodes;
#pragma unroll
      for (int j = 0; j < 6; j++) k[j] = R.rk[j];
    }
    const T xm = side_value<T>(m & 3u, k[0], ph[e + q.xm]);
    const T xp = side_value<T>((m >> 2) & 3u, k[1], ph[e + q.xp]);
    const T ym = side_value<T>((m >> 4) & 3u, k[2], ph[e + q.ym]);
    const T yp = side_value<T>((m >> 6) & 3u, k[3], ph[e + q.yp]);
    const T zm = side_value<T>((m >> 8) & 3u, k[4], ph[e + q.zm]);
    const T zp = side_value<T>((m >> 10) & 3u, k[5], ph[e + q.zp]);
    if (RES && res)
      rh[e] = R.fac * (rh[e] + (xm + xp) * A.rx + (ym + yp) * A.ry + (zm + zp) * A.rz -
                       ph[e] * A.mgparam * R.rdenom);
    else
      ph[e] = (rh[e] + (xm + xp) * A.sx + (ym + yp) * A.sy + (zm + zp) * A.sz) / R.denom +
              A.spm1 * ph[e];
  }
}

// A half sweep of colour c for the dense points of at least the given depth
// (raw: leg_nb).
template <typename T>
__device__ inline void leg_sweep(const LegArgs<T> &A, const LegPts &P, int c, uint32_t depth,
                                 int raw, T *ph, const T *rh) {
  const int ex = A.a[0].ext, sz = ex * A.a[1].ext;
#pragma unroll
  for (int i = 0; i < LEG_NI; i++) {
    const uint32_t p = P.w[i][c];
    if ((p & LEGP_DEPTH) < depth) continue;
    const int e = leg_el(P, i, c);
    const LegNb q = leg_nb(p, ex, sz, raw);
    ph[e] = rh[e] + (ph[e + q.xm] + ph[e + q.xp]) * A.sx + (ph[e + q.ym] + ph[e + q.yp]) * A.sy +
            (ph[e + q.zm] + ph[e + q.zp]) * A.sz + A.spm1 * ph[e];
  }
}

// The tile's phi to memory.
template <typename T>
__device__ inline void leg_store(const LegArgs<T> &A, const LegWin *w, const LegPts &P,
                                 const T *ph, T *__restrict__ out) {
  const int ex = A.a[0].ext, ey = A.a[1].ext, hx = (ex + 1) >> 1;
#pragma unroll
  for (int i = 0; i < LEG_NI; i++) {
    if (!((P.w[i][0] | P.w[i][1]) & LEGP_OWN)) continue;
    const int t = threadIdx.x + i * LEG_TH;
    const int row = leg_div(t, A.mhx), h = t - row * hx;
    const int lz = leg_div(row, A.my), ly = row - lz * ey;
    const int x = w[0].w0 + 2 * h, y = w[1].w0 + ly, z = w[2].w0 + lz;
#pragma unroll
    for (int c = 0; c < 2; c++)
      if (P.w[i][c] & LEGP_OWN)
        out[rb_el(A.g, x + (int)(((P.odd >> i) & 1u) ^ (uint32_t)c), y, z)] =
            ph[leg_el(P, i, c)];
  }
}

template <typename S, typename SC>
__global__ __launch_bounds__(LEG_TH) void k_leg_down(LegArgs<S> A, const S *__restrict__ rho,
                                                     S *__restrict__ phi, SC *__restrict__ rhoc,
                                                     const int *__restrict__ skip) {
  typedef S T;
  typedef typename RestrictArith<S, SC>::type RA;
  extern __shared__ __align__(16) unsigned char leg_lds[];
  // per coarse node and axis: its window's points, their weights and LDS offsets
  __shared__ RA rw[3][LEG_CMAX][5];
  __shared__ int ro[3][LEG_CMAX][5], rn[3][LEG_CMAX];
  const int stop = skip ? *skip : 0;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  const int nt0 = A.a[0].nt, nt1 = A.a[1].nt;
  const LegTile tl[3] = {A.a[0].tile[tile % nt0], A.a[1].tile[tile / nt0 % nt1],
                         A.a[2].tile[tile / (nt0 * nt1)]};
  const int rec0 = A.rec ? (int)A.first[tile] : 0;
  const int nrec = A.rec ? (int)A.first[tile + 1] - rec0 : 0;
  LegRec mq{0u, 0u};
  const int mr = LEG_TH - 1 - (int)threadIdx.x;
  if (mr < nrec) mq = A.rec[rec0 + mr];
  LegWin w[3], b[3], r[3], own[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const LegAxis &a = A.a[k];
    r[k] = leg_clip(a, tl[k].r0, tl[k].r1);
    b[k] = leg_clip(a, tl[k].r0 - 1, tl[k].r1 + 1);
    w[k] = leg_clip(a, tl[k].r0 - 2, tl[k].r1 + 2);
    own[k] = LegWin{tl[k].own0, tl[k].own1};
  }
  const int ex = A.a[0].ext, sz = ex * A.a[1].ext, nw = sz * A.a[2].ext;
  T *ph = reinterpret_cast<T *>(leg_lds), *rh = ph + nw;
  // the restriction's tables on their way (thread i, q: point q of node i)
  const int ti = threadIdx.x / 5, tq = threadIdx.x - 5 * ti;
  double tw[3];
  int tlo[3], thi[3];
  if (ti < LEG_CMAX) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const int c = min(tl[k].c0 + ti, A.a[k].nc);
      tw[k] = A.a[k].rw[5 * c + tq];
      tlo[k] = A.a[k].lo[c];
      thi[k] = A.a[k].hi[c];
    }
  }
  LegPts P;
  leg_load<T, false>(A, w, b, r, own, rho, (const T *)nullptr, ph, rh, P);
  LegRecord<T, true> mine{};
  if (mr < nrec) leg_load_record<T, true>(A, mq, mine);
  if (ti < LEG_CMAX) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const LegAxis &a = A.a[k];
      const int stride = k == 0 ? 1 : k == 1 ? ex : sz;
      int x = tlo[k] + tq;
      // a Neumann guard's residual is its mirror point's
      if (a.bm != 2) x = x < 0 ? -x : x > a.n ? 2 * a.n - x : x;
      rw[k][ti][tq] = (RA)tw[k];
      ro[k][ti][tq] = (x - w[k].w0) * stride;
      if (tq == 0) rn[k][ti] = thi[k] - tlo[k] + 1;
    }
  }
  if (stop) return;  // looked at once the loads are on their way
  // half sweep 0 from phi = 0: a dense point reads its rho alone
#pragma unroll
  for (int i = 0; i < LEG_NI; i++)
    if (P.w[i][0] & LEGP_DEPTH) {
      const int e = leg_el(P, i, 0);
      const T o = (T)0.;
      ph[e] = rh[e] + (o + o) * A.sx + (o + o) * A.sy + (o + o) * A.sz + A.spm1 * o;
    }
  __syncthreads();
  if (nrec) {
    // (records read only their own rho and phi here: written above by other
    // threads, hence the barrier)
    leg_records<T, true>(A, w, w, 0, false, true, 0, ph, rh, rec0, nrec, mine);
    __syncthreads();
  }
  leg_sweep<T>(A, P, 1, 2u, 0, ph, rh);
  if (nrec) leg_records<T, true>(A, w, b, 1, false, false, 0, ph, rh, rec0, nrec, mine);
  __syncthreads();
  leg_store<T>(A, w, P, ph, phi);
  // the residual, in the place of rho (each point reads its own rho alone)
#pragma unroll
  for (int i = 0; i < LEG_NI; i++)
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const uint32_t p = P.w[i][c];
      if (p & LEGP_INT) rh[leg_el(P, i, c)] = (T)0.;
      if ((p & LEGP_DEPTH) < 3u) continue;
      const int e = leg_el(P, i, c);
      const LegNb q = leg_nb(p, ex, sz, 0);
      rh[e] = rh[e] + (ph[e + q.xm] + ph[e + q.xp]) * A.rx + (ph[e + q.ym] + ph[e + q.yp]) * A.ry +
              (ph[e + q.zm] + ph[e + q.zp]) * A.rz - ph[e] * A.mgparam;
    }
  if (nrec)
#pragma unroll 1
    for (int c = 0; c < 2; c++)
      leg_records<T, true>(A, w, r, c, true, false, 0, ph, rh, rec0, nrec, mine);
  __syncthreads();
  // restriction (restrict_point, k_restrict_t)
  const int nx = tl[0].c1 - tl[0].c0 + 1, ny = tl[1].c1 - tl[1].c0 + 1,
            nz = tl[2].c1 - tl[2].c0 + 1;
  for (int t = threadIdx.x; t < nx * ny * nz; t += LEG_TH) {
    const int ix = t % nx, u0 = t / nx, iy = u0 % ny, iz = u0 / ny;
    RA s = (RA)0., u = (RA)0.;
    if (A.plain) {
      const T *o = rh + ro[0][ix][0] + ro[1][iy][0] + ro[2][iz][0];
      T v[27];
#pragma unroll
      for (int q = 0; q < 27; q++) v[q] = o[q % 3 + ex * ((q / 3) % 3) + sz * (q / 9)];
      RA wxy[9];
#pragma unroll
      for (int q = 0; q < 9; q++) wxy[q] = rw[0][ix][q % 3] * rw[1][iy][q / 3];
#pragma unroll
      for (int q = 0; q < 27; q++) {
        const RA ww = wxy[q % 9] * rw[2][iz][q / 9];
        s = s + ww * (RA)v[q];
        u = u + ww;
      }
    } else {
      const int mx = rn[0][ix], my = rn[1][iy], mz = rn[2][iz];
#pragma unroll 1
      for (int kz = 0; kz < mz; kz++)
#pragma unroll 1
        for (int ky = 0; ky < my; ky++) {
          const RA wy = rw[1][iy][ky], wz = rw[2][iz][kz];
          const T *row = rh + ro[1][iy][ky] + ro[2][iz][kz];
#pragma unroll
          for (int kx = 0; kx < 5; kx++)
            if (kx < mx) {
              const RA ww = rw[0][ix][kx] * wy * wz;
              s = s + ww * (RA)row[ro[0][ix][kx]];
              u = u + ww;
            }
        }
    }
    rhoc[rb_el(A.gc, tl[0].c0 + ix, tl[1].c0 + iy, tl[2].c0 + iz)] =
        u > (RA)0. ? (SC)((s / u) * (RA)A.ff) : (SC)0.;
  }
}

template <typename S, typename SC>
__global__ __launch_bounds__(LEG_TH) void k_leg_up(LegArgs<S> A, const S *__restrict__ rho,
                                                   const S *__restrict__ phi,
                                                   const SC *__restrict__ phic,
                                                   S *__restrict__ out,
                                                   const int *__restrict__ skip) {
  typedef S T;
  extern __shared__ __align__(16) unsigned char leg_lds[];
  __shared__ T ew[3][LEG_WMAX];
  __shared__ int ej[3][LEG_WMAX];
  const int stop = skip ? *skip : 0;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  const int nt0 = A.a[0].nt, nt1 = A.a[1].nt;
  const LegTile tl[3] = {A.a[0].tile[tile % nt0], A.a[1].tile[tile / nt0 % nt1],
                         A.a[2].tile[tile / (nt0 * nt1)]};
  const int rec0 = A.rec ? (int)A.first[tile] : 0;
  const int nrec = A.rec ? (int)A.first[tile + 1] - rec0 : 0;
  LegRec mq{0u, 0u};
  const int mr = LEG_TH - 1 - (int)threadIdx.x;
  if (mr < nrec) mq = A.rec[rec0 + mr];
  LegWin w[3], c[3], own[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const LegAxis &a = A.a[k];
    own[k] = LegWin{tl[k].own0, tl[k].own1};
    c[k] = leg_clip(a, own[k].w0 - 1, own[k].w1 + 1);
    w[k] = leg_clip(a, own[k].w0 - 2, own[k].w1 + 2);
  }
  const int ex = A.a[0].ext, ey = A.a[1].ext, nw = ex * ey * A.a[2].ext, hx = (ex + 1) >> 1;
  const int fx = A.a[0].cext, fy = A.a[1].cext, fz = fx * fy, nq = fz * A.a[2].cext;
  T *ph = reinterpret_cast<T *>(leg_lds), *rh = ph + nw, *pc = rh + nw;
  // the expansion's tables and the coarse phi on their way
  const int ti = threadIdx.x;
  double tw[3];
  int tj[3];
  if (ti < LEG_WMAX) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const LegAxis &a = A.a[k];
      const int x = min(w[k].w0 + ti, w[k].w1), u = leg_wrap(a, x);
      const int run = a.bm != 2 ? 0 : x < 0 ? -a.nc : x >= a.n ? a.nc : 0;
      tj[k] = a.ej[u] + run - tl[k].c0;
      tw[k] = a.ew[u];
    }
  }
  constexpr int QN = 2;  // coarse points per thread in flight
  T cv[QN];
  auto coarse = [&](int t) {
    const int row = leg_div(t, A.mcx), lx = t - row * fx;
    const int lz = leg_div(row, A.mcy), ly = row - lz * fy;
    // beyond a Neumann face the weight is zero: any value of the level does
    auto in = [](const LegAxis &a, int i) {
      if (a.bm != 2) return min(i, a.nc);
      return i < 0 ? i + a.nc : i > a.nc ? i - a.nc : i;
    };
    return (T)phic[rb_el(A.gc, in(A.a[0], min(tl[0].c0 + lx, tl[0].c1)),
                         in(A.a[1], min(tl[1].c0 + ly, tl[1].c1)),
                         in(A.a[2], min(tl[2].c0 + lz, tl[2].c1)))];
  };
#pragma unroll
  for (int k = 0; k < QN; k++) cv[k] = coarse(min(ti + k * LEG_TH, nq - 1));
  LegPts P;
  leg_load<T, true>(A, w, c, own, own, rho, phi, ph, rh, P);
#pragma unroll
  for (int k = 0; k < QN; k++)
    if (ti + k * LEG_TH < nq) pc[ti + k * LEG_TH] = cv[k];
  for (int t = ti + QN * LEG_TH; t < nq; t += LEG_TH) pc[t] = coarse(t);
  LegRecord<T, false> mine{};
  if (mr < nrec) leg_load_record<T, false>(A, mq, mine);
  if (ti < LEG_WMAX) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
      ej[k][ti] = tj[k] * (k == 0 ? 1 : k == 1 ? fx : fz);
      ew[k][ti] = (T)tw[k];
    }
  }
  if (stop) return;  // looked at once the loads are on their way
  __syncthreads();
  // expansion (k_expand_rb), and the pin of the interior points; a record's
  // point is expanded by the thread of its pair as well
#pragma unroll
  for (int i = 0; i < LEG_NI; i++) {
    if (P.e[i] < 0) continue;
    const int t = threadIdx.x + i * LEG_TH;
    const int row = leg_div(t, A.mhx), h = t - row * hx;
    const int lz = leg_div(row, A.my), ly = row - lz * ey;
    const T one = (T)1., wy = ew[1][ly], wz = ew[2][lz];
    const T *oyz = pc + ej[1][ly] + ej[2][lz];
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const uint32_t p = P.w[i][q];
      if (!(p & (LEGP_DEPTH | LEGP_INT | LEGP_REC))) continue;
      const int dx = (int)(((P.odd >> i) & 1u) ^ (uint32_t)q), e = P.e[i] + dx;
      const T wx = ew[0][2 * h + dx];
      const T *o = oyz + ej[0][2 * h + dx];
      const T v = ph[e] + (one - wx) * (one - wy) * (one - wz) * o[0] +
                  wx * (one - wy) * (one - wz) * o[1] + (one - wx) * wy * (one - wz) * o[fx] +
                  wx * wy * (one - wz) * o[fx + 1] + (one - wx) * (one - wy) * wz * o[fz] +
                  wx * (one - wy) * wz * o[fz + 1] + (one - wx) * wy * wz * o[fz + fx] +
                  wx * wy * wz * o[fz + fx + 1];
      ph[e] = p & LEGP_INT ? (T)0. : v;
      if (p & LEGP_INT) rh[e] = v;  // (before the pin: leg_nb's raw)
    }
  }
  __syncthreads();
  leg_sweep<T>(A, P, 0, 2u, nw, ph, rh);
  if (nrec) leg_records<T, false>(A, w, c, 0, false, false, nw, ph, rh, rec0, nrec, mine);
  __syncthreads();
  leg_sweep<T>(A, P, 1, 3u, 0, ph, rh);
  if (nrec) leg_records<T, false>(A, w, own, 1, false, false, 0, ph, rh, rec0, nrec, mine);
  __syncthreads();
  leg_store<T>(A, w, P, ph, out);
}
