// The coarse end of the FP64 V-cycle in one launch.  Included by mg3d.hip.
//
// On the small coarse levels (a few thousand nodes) each step of vcycle
// (f3d_mgrid.F:1101-1591) -- a half sweep, the residual, the restriction,
// the expansion -- is a launch of a few microseconds whose time is launch
// latency and the z-march's serial chain, not bytes.  k_vtail runs the
// whole V-cycle from a level T down to the coarsest and back in one
// workgroup of 1024 threads: every step becomes a phase in which the
// threads stride over the step's points, and phases are separated by
// workgroup barriers.  The levels' phi, rho and res live in LDS for the
// whole launch, in the same red-black layout and element numbering as
// their HBM arrays (these levels' rows are not padded), and so do the
// read-only tables the steps use (points to update, conductor records'
// constants, transfer windows and weights).  The launch starts by copying an
// image of the tables from HBM, 16 bytes per lane with every load in flight
// (k_tail_image gathers it once per solve), and level T's rho, and zeroes the
// level arrays meanwhile.  At its end it writes level T's phi back; between
// the two every phase reads and writes LDS only.
//
// A phase costs latency and instructions of waves that find nothing to do, so:
// the points of a half sweep and of the residual come from a table of words
// (element, row parity, faces), decoded once per solve; a pass's numbers are
// one record, read at the start of the launch so that the scalar cache holds
// it; and there are as few phases as possible.  Where the interior points
// allow it (TAIL_WRAP) the neighbours across a Neumann or periodic face are
// found by address, which leaves out the boundary conditions and the pins
// after them (on a periodic axis the ranges end at n - 1 and who writes plane
// 0 writes plane n too); the zeros of the residual are the launch's.
//
// Measured (one launch, cycles of 2.3 GHz; before: points decoded in each
// phase, all of LDS gathered, boundary and pin phases): 64x64x64 without
// conductors (levels from 8x8x16) 78k -> 49k, of which a half sweep 1.3k and
// the start 14k (three memory round trips); 128x128x256 with the pipe and the
// annulus 115k -> 85k; with periodic ends and quadrupoles 193k -> 103k (its
// solve 20.2 -> 16.9 ms with the level above it as legs); 101x75x190 with
// Neumann faces 208k -> 86k.
//
// Each phase evaluates its points with the arithmetic of the kernel it
// replaces (the same device functions where they exist, the same
// expressions in the same order otherwise), and the phases follow the
// launch order of the host path (sorpass, residual_rb, restrict_to,
// expand_rb and their boundary conditions), so the results are the same
// bits.
#pragma once
#include "mg3d_kernels.h"

enum {
  TAIL_PIN_AFTER = 1,  // pin (and mirror) after every half sweep
  TAIL_MIRROR = 2,     // Neumann subgrid mirrors after each pin
  TAIL_PER = 4,        // TAIL_WRAP with a periodic axis
  TAIL_FUSEPIN = 8,    // the expansion into this level writes the first up pass's pin
  TAIL_GUARD = 16,     // the expansion writes the guard points, from values before the pin
  TAIL_RES1 = 32,      // the residual's records can share the dense phase
  TAIL_WRAP = 64,      // neighbours across faces by address, no boundary phases
  TAIL_HALF = 128,     // restriction windows [2j-1, 2j+1] in every axis, at the faces too
};

// A point's word: its element within its colour, ix even, the faces it lies
// on across which its neighbour is found by address (x low, x high, y ...),
// the periodic axes in which it is on plane 0 and stands for plane n too.
enum { TW_EVEN = 1 << 16, TW_FACE = 1 << 17, TW_IMAGE = 1 << 23 };
constexpr uint32_t TW_NONE = 1u << 31;  // nothing to do

// A half sweep or residual of one colour: LDS word offsets of the colour's
// arrays, the points' table, the records.
struct TailPass {
  int n, tab;              // dense points
  int own, oth, rho, dst;  // phi of the colour and of the other one, rho, result
  int W, pl;               // elements of a row and of a plane
  int f[6];                // elements to the neighbours across the faces
  int im[3];               // elements to the images
  int res;                 // residual
  int nr, rtab, modes, k, denom, fac;
  double c[4];             // coefficients of the dense points: x, y, z, own
  double r[4];             // and of the records (own: 1 - mgparam or mgparam)
};

// A record list in LDS: word offsets of the SubList arrays.
struct TailSub {
  int n, pos, modes, k, denom, fac, zero;
};
// Restriction and expansion tables in LDS (word offsets) with their ranges.
struct TailAxisR {
  int lo, hi, w, cmin, cmax;
};
struct TailAxisE {
  int j, w, lo, hi;
};

// One level of the tail, built on the host.  Offsets count 32-bit words of
// the launch's LDS; arrays of doubles start at even offsets.
struct TailLevel {
  RBGeom g;
  double *phi;              // HBM phi (the first level's is written back)
  int lphi, lrho, lres;     // phi, rho, res
  int limask, lint;         // imask words, interior positions
  double rs[3];             // coefficients of the record residuals
  TailSub rsub[2];          // records of the residual (without TAIL_RES1)
  int nint, flags;
  int nsub[2];              // Neumann mirror lists (condbndymgint), read from HBM
  const int *subpos[2];
  const double *subdels[2];
  TailAxisR ra[3];          // restriction to the next level
  double ff;
  TailAxisE ea[3];          // expansion from the next level
  uint32_t mr[2], me[2];    // reciprocals of the decoding divisors of both
};

// A part of the image: words dst.. of the LDS, copied from HBM or made.
enum { TIM_COPY = 0, TIM_POINTS = 1, TIM_RECORDS = 2 };
struct TailItem {
  const uint32_t *src;  // the array, the mask (or NULL), the records' positions
  int dst, words, kind, colour;
  RBGeom g;
  int r[6];             // the range of the points
  int b[6];             // bounds across which neighbours are found by address (else 0)
};

constexpr int TAIL_MAX_ITEMS = 256;

// The launch runs a list of steps built on the host in the order the host
// path would launch them (each step's code appears once in the kernel, so
// the kernel stays small enough for the instruction cache).
enum {
  TOP_PIN = 0,       // cond_potmg (+ condbndymgint)
  TOP_PASS = 1,      // half sweep or residual of one colour: pass `pass`
  TOP_BCPHI = 2,     // boundary conditions on phi
  TOP_RESREC = 3,    // the residual's records where they need an order
  TOP_BCRES = 4,     // boundary conditions on the residual
  TOP_RESTRICT = 5,  // restriction to level+1
  TOP_EXPAND = 6,    // expansion from level+1 (with its boundary conditions)
};
// arg of TOP_PASS
enum { TPASS_FACES = 1, TPASS_SYNC = 2 };
struct TailOp {
  int kind, level, arg, pass;
};

constexpr int TAIL_MAX_OPS = 1024;

struct TailRun {
  int nops;
  int at_pass, at_level, desc_bytes;  // the steps, passes and levels in one buffer
  int b[6];
  double mgparam;
  int tab_words, lds_words;  // LDS of the tables and in all (32-bit words, multiples of four)
  const uint32_t *image;
  const uint32_t *rho0;  // the first level's rho, to words lrho0..
  int lrho0, rho_words;
};

#define TAIL_FOR(t, n) for (int t = (int)threadIdx.x; t < (int)(n); t += (int)blockDim.x)

__device__ inline bool tail_bit(const uint32_t *m, int e) { return (m[e >> 5] >> (e & 31)) & 1u; }

__device__ inline double *tail_d(uint32_t *w, int off) { return reinterpret_cast<double *>(w + off); }

__device__ inline SubList<double> tail_sub(const TailSub &s, uint32_t *w) {
  return SubList<double>{s.n, reinterpret_cast<const int *>(w + s.pos), w + s.modes,
                         tail_d(w, s.k), tail_d(w, s.denom), tail_d(w, s.fac), w + s.zero};
}

__device__ inline RestrictAxis tail_ra(const TailAxisR &a, uint32_t *w) {
  return RestrictAxis{reinterpret_cast<const int *>(w + a.lo),
                      reinterpret_cast<const int *>(w + a.hi), tail_d(w, a.w), a.cmin, a.cmax};
}

__device__ inline ExpandAxis tail_ea(const TailAxisE &a, uint32_t *w) {
  return ExpandAxis{reinterpret_cast<const int *>(w + a.j), tail_d(w, a.w), a.lo, a.hi};
}

__device__ inline const int *tail_int(const TailLevel &L, uint32_t *w) {
  return reinterpret_cast<const int *>(w + L.lint);
}

// cond_potmg without voltages (k_pin) and condbndymgint (k_condbndymgint).
__device__ inline void tail_pin(const TailLevel &L, const TailRun &R, uint32_t *w) {
  double *phi = tail_d(w, L.lphi);
  const int *ip = tail_int(L, w);
  TAIL_FOR(i, L.nint) { phi[rb_index(L.g, ip[3 * i], ip[3 * i + 1], ip[3 * i + 2])] = 0.; }
  __syncthreads();
  if (L.flags & TAIL_MIRROR) {
    if (threadIdx.x == 0)
      condbndymgint_seq<double>(phi, L.g, L.nsub[0], L.nsub[1], L.subpos[0], L.subpos[1],
                                L.subdels[0], L.subdels[1], R.b[0], R.b[1], R.b[2], R.b[3],
                                R.b[4], R.b[5]);
    __syncthreads();
  }
}

// applyboundaryconditions3d without Dirichlet guards (k_bc_axis, x then y
// then z; axes whose two bounds are Dirichlet change nothing).
__device__ inline void tail_bc(double *u, const RBGeom &g, const TailRun &R) {
  for (int a = 0; a < 3; a++) {
    if (R.b[2 * a] == 0 && R.b[2 * a + 1] == 0) continue;
    const int na = a == 0 ? g.ny : g.nx, nb = a == 2 ? g.ny : g.nz;
    TAIL_FOR(t, (na + 3) * (nb + 3)) {
      bc_line<double, RBIdx>(u, RBIdx{g}, a, g.nx, g.ny, g.nz, R.b[2 * a], R.b[2 * a + 1], 0, 0,
                             t);
    }
    __syncthreads();
  }
}

// The word of the point (ix, iy, iz).
__device__ inline uint32_t tail_word(const RBGeom &g, const int *b, int ix, int iy, int iz) {
  uint32_t d = (uint32_t)(g.W * (iy + 1 + g.PY * (iz + 1)) + ((ix + 1) >> 1));
  if (!(ix & 1)) d |= TW_EVEN;
  const int i[3] = {ix, iy, iz}, n[3] = {g.nx, g.ny, g.nz};
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (b[2 * a] == 2 && i[a] == n[a]) return TW_NONE;  // an image
    if (b[2 * a] && i[a] == 0) d |= TW_FACE << (2 * a);
    if (b[2 * a + 1] && i[a] == n[a]) d |= TW_FACE << (2 * a + 1);
    if (b[2 * a] == 2 && i[a] == 0) d |= TW_IMAGE << a;
  }
  return d;
}

// The image of the launch's tables, each block an item (every solve: an
// item's array may have new contents).
__global__ __launch_bounds__(256) void k_tail_image(const TailItem *__restrict__ items,
                                                    uint32_t *__restrict__ image) {
  const TailItem &it = items[blockIdx.x];
  const int *r = it.r;
  const int j0 = (r[0] + 1) / 2, nj = (r[1] + 1) / 2 - j0 + 1, ny = r[3] - r[2] + 1;
  for (int k = threadIdx.x; k < it.words; k += 256) {
    uint32_t v;
    if (it.kind == TIM_COPY) {
      v = it.src[k];
    } else if (it.kind == TIM_RECORDS) {
      const int *q = reinterpret_cast<const int *>(it.src) + 3 * k;
      v = tail_word(it.g, it.b, q[0], q[1], q[2]);
    } else {
      const int j = j0 + k % nj, u = k / nj, iy = r[2] + u % ny, iz = r[4] + u / ny;
      const int ix = 2 * j - 1 + ((it.colour + iy + iz + 1) & 1);
      const int ce = it.colour * (int)it.g.cs + it.g.W * (iy + 1 + it.g.PY * (iz + 1)) + j;
      const bool skip = ix < r[0] || ix > r[1] ||
                        (it.src && ((it.src[ce >> 5] >> (ce & 31)) & 1u));
      v = skip ? TW_NONE : tail_word(it.g, it.b, ix, iy, iz);
    }
    image[it.dst + k] = v;
  }
}

// Elements of the six neighbours of a word's point, all of the other colour.
struct TailNb {
  int xm, xp, ym, yp, zm, zp;
};

__device__ inline TailNb tail_nb(const TailPass &p, uint32_t d, uint32_t faces) {
  const int e = (int)(d & 0xffffu), x = e + (int)((d >> 16) & 1u);
  TailNb q{x - 1, x, e - p.W, e + p.W, e - p.pl, e + p.pl};
  if (d & faces) {
    if (d & (TW_FACE << 0)) q.xm = e + p.f[0];
    if (d & (TW_FACE << 1)) q.xp = e + p.f[1];
    if (d & (TW_FACE << 2)) q.ym = e + p.f[2];
    if (d & (TW_FACE << 3)) q.yp = e + p.f[3];
    if (d & (TW_FACE << 4)) q.zm = e + p.f[4];
    if (d & (TW_FACE << 5)) q.zp = e + p.f[5];
  }
  return q;
}

// A pass's result at a word's point, and at its images.
__device__ inline void tail_store(const TailPass &p, double *u, uint32_t d, double v) {
  const int e = (int)(d & 0xffffu);
  u[e] = v;
  if (!(d & (7u * TW_IMAGE))) return;
#pragma unroll 1
  for (uint32_t m = 1; m < 8; m++)
    if (((d / TW_IMAGE) & m) == m)
      u[e + (m & 1 ? p.im[0] : 0) + (m & 2 ? p.im[1] : 0) + (m & 4 ? p.im[2] : 0)] = v;
}

// One half sweep of a colour, or its residual: the dense points as
// k_sor_zmarch and k_residual_pairs update them and the colour's records
// (sor_record, residual_record); all write different points and read the
// other colour and their own values only.  faces: neighbours across the faces
// by address (else from the guard points).
__device__ inline void tail_pass(const TailPass &p, bool by_address, uint32_t *w) {
  const uint32_t faces = by_address ? 63u * TW_FACE : 0u;
  const double *o = tail_d(w, p.oth), *own = tail_d(w, p.own), *rho = tail_d(w, p.rho);
  double *dst = tail_d(w, p.dst);
  const uint32_t *tab = w + p.tab;
  TAIL_FOR(t, p.n) {
    const uint32_t d = tab[t];
    if (d & TW_NONE) continue;
    const int e = (int)(d & 0xffffu);
    const TailNb q = tail_nb(p, d, faces);
    tail_store(p, dst, d,
               rho[e] + (o[q.xm] + o[q.xp]) * p.c[0] + (o[q.ym] + o[q.yp]) * p.c[1] +
                   (o[q.zm] + o[q.zp]) * p.c[2] + own[e] * p.c[3]);
  }
  // (the last threads first: they have the fewest points)
  for (int i = (int)blockDim.x - 1 - (int)threadIdx.x; i < p.nr; i += (int)blockDim.x) {
    const uint32_t d = w[p.rtab + i];
    if (d & TW_NONE) continue;
    const int e = (int)(d & 0xffffu);
    const TailNb q = tail_nb(p, d, faces);
    const uint32_t m = w[p.modes + i];
    const double *k = tail_d(w, p.k) + 6 * i;
    const double denom = tail_d(w, p.denom)[i];
    const double xm = side_value<double>(m & 3u, k[0], o[q.xm]);
    const double xp = side_value<double>((m >> 2) & 3u, k[1], o[q.xp]);
    const double ym = side_value<double>((m >> 4) & 3u, k[2], o[q.ym]);
    const double yp = side_value<double>((m >> 6) & 3u, k[3], o[q.yp]);
    const double zm = side_value<double>((m >> 8) & 3u, k[4], o[q.zm]);
    const double zp = side_value<double>((m >> 10) & 3u, k[5], o[q.zp]);
    const double s = rho[e] + (xm + xp) * p.r[0] + (ym + yp) * p.r[1] + (zm + zp) * p.r[2];
    tail_store(p, dst, d,
               p.res ? tail_d(w, p.fac)[i] * (s - own[e] * p.r[3] * denom)
                     : s / denom + p.r[3] * own[e]);
  }
}

// The residual's records where one zeroes a neighbour's residual or sits on an
// interior point: the lists in order, as the host launches them.
__device__ inline void tail_residual_records(const TailLevel &L, const TailRun &R, uint32_t *w) {
  const RBGeom g = L.g;
  const double *phi = tail_d(w, L.lphi), *rho = tail_d(w, L.lrho);
  double *res = tail_d(w, L.lres);
#pragma unroll 1
  for (int p = 0; p < 2; p++) {
    const SubList<double> sub = tail_sub(L.rsub[p], w);
    if (sub.n == 0) continue;
    TAIL_FOR(i, sub.n) {
      residual_record<double, double, double, RBIdx>(phi, rho, res, RBIdx{g}, g, sub, i, L.rs[0],
                                                     L.rs[1], L.rs[2], R.mgparam);
    }
    __syncthreads();
  }
}

// t / d with d's reciprocal m (t d < 2^32).
__device__ inline int tail_div(int t, int d, uint32_t m) {
  return d == 1 ? t : (int)__umulhi((uint32_t)t, m);
}

// A coordinate's image inside the level.
__device__ inline int tail_in(int i, int n, int bm, int bp) {
  if (i < 0) return bm == 1 ? -i : i + n;
  if (i > n) return bp == 1 ? 2 * n - i : i - n;
  return i;
}

// restrict3d of L's residual into the source of the next level C
// (restrict_point).  C's phi is zero already: nothing has written it.  With
// TAIL_WRAP a guard point's residual is its image's.
__device__ inline void tail_restrict(const TailLevel &L, const TailLevel &C, const TailRun &R,
                                     uint32_t *w) {
  const RBGeom gc = C.g, g = L.g;
  const double *res = tail_d(w, L.lres);
  double *rhoc = tail_d(w, C.lrho);
  const RestrictAxis ax = tail_ra(L.ra[0], w), ay = tail_ra(L.ra[1], w), az = tail_ra(L.ra[2], w);
  const int mx = ax.cmax - ax.cmin + 1, my = ay.cmax - ay.cmin + 1, mz = az.cmax - az.cmin + 1;
  const bool wrap = L.flags & TAIL_WRAP;
  const int W = g.W, pl = g.W * g.PY, cs = (int)g.cs;
  TAIL_FOR(t, mx * my * mz) {
    const int u0 = tail_div(t, mx, L.mr[0]), u1 = tail_div(u0, my, L.mr[1]);
    const int ixc = ax.cmin + t - mx * u0, iyc = ay.cmin + u0 - my * u1, izc = az.cmin + u1;
    double r = 0.;
    if (L.flags & TAIL_HALF) {
      // the weights are 1/2, 1, 1/2 and sum up to 8, exactly
      int xe[3], ro[3], po[3];
#pragma unroll
      for (int k = 0; k < 3; k++) {
        int x = 2 * ixc - 1 + k, y = 2 * iyc - 1 + k, z = 2 * izc - 1 + k;
        if (wrap) {  // (the images have the same parity)
          x = tail_in(x, g.nx, R.b[0], R.b[1]);
          y = tail_in(y, g.ny, R.b[2], R.b[3]);
          z = tail_in(z, g.nz, R.b[4], R.b[5]);
        }
        xe[k] = (x + 1) >> 1;
        ro[k] = W * (y + 1);
        po[k] = pl * (z + 1);
      }
      double v[27];
#pragma unroll
      for (int q = 0; q < 27; q++) {
        const int c = (q + 1) & 1;  // the colour: parity of the coordinates' sum
        v[q] = res[po[q / 9] + ro[(q / 3) % 3] + xe[q % 3] + (c ? cs : 0)];
      }
#pragma unroll
      for (int q = 0; q < 27; q++) {
        const double ww = (q % 3 == 1 ? 1. : 0.5) * ((q / 3) % 3 == 1 ? 1. : 0.5) *
                          (q / 9 == 1 ? 1. : 0.5);
        r = r + ww * v[q];
      }
      rhoc[rb_el(gc, ixc, iyc, izc)] = (r / 8.) * L.ff;
      continue;
    }
    const double *wx = ax.w + 5 * ixc, *wy = ay.w + 5 * iyc, *wz = az.w + 5 * izc;
    double s = 0.;
    const int x0 = ax.lo[ixc], nx = ax.hi[ixc] - x0, y0 = ay.lo[iyc], y1 = ay.hi[iyc];
    const int z0 = az.lo[izc], z1 = az.hi[izc];
    int xe[5], xc[5];  // a window's elements, and with the colour for rows of even y + z
    double wxk[5];
#pragma unroll
    for (int k = 0; k < 5; k++) {
      int x = x0 + min(k, nx);
      if (wrap) x = tail_in(x, g.nx, R.b[0], R.b[1]);
      xe[k] = (x + 1) >> 1;
      xc[k] = x & 1 ? cs : 0;
      wxk[k] = wx[k];
    }
#pragma unroll 1
    for (int iz = z0; iz <= z1; iz++)
#pragma unroll 1
      for (int iy = y0; iy <= y1; iy++) {
        const double wyq = wy[iy - y0], wzq = wz[iz - z0];
        const int fy = wrap ? tail_in(iy, g.ny, R.b[2], R.b[3]) : iy,
                  fz = wrap ? tail_in(iz, g.nz, R.b[4], R.b[5]) : iz;
        const int row = W * (fy + 1) + pl * (fz + 1), odd = (fy + fz) & 1 ? cs : 0;
        double v[5];
#pragma unroll
        for (int k = 0; k < 5; k++) v[k] = res[row + xe[k] + (xc[k] ^ odd)];
#pragma unroll
        for (int k = 0; k < 5; k++)
          if (k <= nx) {
            const double ww = wxk[k] * wyq * wzq;
            r = r + ww * v[k];
            s = s + ww;
          }
      }
    rhoc[rb_el(gc, ixc, iyc, izc)] = s > 0. ? (r / s) * L.ff : 0.;
  }
  __syncthreads();
}

// The images of an expanded point on the planes n of periodic axes, and (with
// TAIL_GUARD) its guard points, which hold the value from before the pin: the
// boundary conditions run between the expansion and the pin.
template <typename F>
__device__ inline void tail_expand_faces(const TailLevel &L, const TailRun &R, double *phi, int e,
                                         int ix, int iy, int iz, double v, const F &put) {
  const RBGeom &g = L.g;
  const int i[3] = {ix, iy, iz}, n[3] = {g.nx, g.ny, g.nz}, st[3] = {1, 2 * g.W, 2 * g.W * g.PY};
  int off[3];  // to the image, in elements (0: none)
#pragma unroll
  for (int a = 0; a < 3; a++) {
    off[a] = R.b[2 * a] == 2 && i[a] == 0 ? st[a] * (n[a] >> 1) : 0;
    if (!(L.flags & TAIL_GUARD)) continue;
    if (R.b[2 * a] == 1 && i[a] == 1) phi[e - st[a]] = v;
    if (R.b[2 * a + 1] == 1 && i[a] == n[a] - 1) phi[e + st[a]] = v;
    if (R.b[2 * a] == 2 && i[a] == n[a] - 1) phi[e - st[a] * (n[a] >> 1)] = v;
  }
  if (!(off[0] | off[1] | off[2])) return;
#pragma unroll 1
  for (int m = 1; m < 8; m++) {
    if (((m & 1) && !off[0]) || ((m & 2) && !off[1]) || ((m & 4) && !off[2])) continue;
    put(e + (m & 1 ? off[0] : 0) + (m & 2 ? off[1] : 0) + (m & 4 ? off[2] : 0));
  }
}

// expand3d of C's phi added to L's (the sum of k_expand_rb, term for term),
// with the pin of the first up pass where it is fused, then the boundary
// conditions.
__device__ inline void tail_expand(const TailLevel &L, const TailLevel &C, const TailRun &R,
                                   uint32_t *w) {
  const ExpandAxis ax = tail_ea(L.ea[0], w), ay = tail_ea(L.ea[1], w), az = tail_ea(L.ea[2], w);
  const int nxr = ax.hi - ax.lo + 1, nyr = ay.hi - ay.lo + 1, nzr = az.hi - az.lo + 1;
  const bool fusepin = L.flags & TAIL_FUSEPIN;
  double *phi = tail_d(w, L.lphi);
  if (nxr <= 0 || nyr <= 0 || nzr <= 0) {
    if (fusepin) tail_pin(L, R, w);
  } else {
    const RBGeom g = L.g, gc = C.g;
    const double *pc = tail_d(w, C.lphi);
    const uint32_t *imask = w + L.limask;
    const double one = 1.;
    TAIL_FOR(t, nxr * nyr * nzr) {
      const int u0 = tail_div(t, nxr, L.me[0]), u1 = tail_div(u0, nyr, L.me[1]);
      const int ix = ax.lo + t - nxr * u0, iy = ay.lo + u0 - nyr * u1, iz = az.lo + u1;
      const int jx = ax.j[ix], jy = ay.j[iy], jz = az.j[iz];
      const double wx = ax.w[ix], wy = ay.w[iy], wz = az.w[iz];
      const int e = rb_el(g, ix, iy, iz);
      // the coarse cell: the elements of its two x in rows of its first row's
      // parity (a) and of the other (b)
      const int row = gc.W * (jy + 1 + gc.PY * (jz + 1)), cp = gc.W * gc.PY;
      const int odd = (jx + jy + jz) & 1 ? (int)gc.cs : 0, even = (int)gc.cs - odd;
      const int e0 = row + ((jx + 1) >> 1), e1 = row + ((jx + 2) >> 1);
      const int a0 = e0 + odd, a1 = e1 + even, b0 = e0 + even, b1 = e1 + odd;
      const double v = phi[e] + (one - wx) * (one - wy) * (one - wz) * pc[a0] +
                       wx * (one - wy) * (one - wz) * pc[a1] +
                       (one - wx) * wy * (one - wz) * pc[b0 + gc.W] +
                       wx * wy * (one - wz) * pc[b1 + gc.W] +
                       (one - wx) * (one - wy) * wz * pc[b0 + cp] +
                       wx * (one - wy) * wz * pc[b1 + cp] +
                       (one - wx) * wy * wz * pc[a0 + gc.W + cp] +
                       wx * wy * wz * pc[a1 + gc.W + cp];
      auto put = [&](int k) { phi[k] = (fusepin && tail_bit(imask, k)) ? 0. : v; };
      put(e);
      if (L.flags & (TAIL_PER | TAIL_GUARD)) tail_expand_faces(L, R, phi, e, ix, iy, iz, v, put);
    }
    __syncthreads();
  }
  if (!(L.flags & TAIL_WRAP)) tail_bc(phi, L.g, R);
}

// Reads a table once, sixteen lines in flight, so that the scalar cache holds it.
__device__ inline void tail_touch(const void *p, int bytes) {
  const int *a = (const int *)p;
  const int n = bytes / 64;
  for (int k = 0; k < n; k += 16) {
    int s = 0;
#pragma unroll
    for (int j = 0; j < 16; j++) s |= a[16 * min(k + j, n - 1)];
    asm volatile("" ::"s"(s));
  }
}

// The V-cycle from tl[0] (whose phi starts at zero) to the coarsest level
// and back, as the list of steps ops.
__global__ __launch_bounds__(1024) void k_vtail(const unsigned char *__restrict__ desc, TailRun R,
                                                const int *__restrict__ skip) {
  // the steps, passes and levels one after the other
  const TailOp *ops = (const TailOp *)desc;
  const TailPass *passes = (const TailPass *)(desc + R.at_pass);
  const TailLevel *tl = (const TailLevel *)(desc + R.at_level);
  extern __shared__ __align__(16) uint32_t tail_lds[];
  uint32_t *w = tail_lds;
  const int stop = skip ? *skip : 0;
  // the tables and the first level's rho, all loads before the stores
  constexpr int NI = 6, NR = 8;
  const uint4 *img = (const uint4 *)R.image;
  uint4 v[NI];
  uint32_t q[NR];
  const int n4 = R.tab_words / 4;
#pragma unroll
  for (int k = 0; k < NI; k++) {
    const int t = (int)threadIdx.x + 1024 * k;
    if (t < n4) v[k] = img[t];
  }
#pragma unroll
  for (int k = 0; k < NR; k++) {
    const int t = (int)threadIdx.x + 1024 * k;
    if (t < R.rho_words) q[k] = R.rho0[t];
  }
  // (the steps' numbers to L2, a line per lane)
  if ((int)threadIdx.x < R.desc_bytes / 64) {
    const int x = ((const int *)desc)[16 * threadIdx.x];
    asm volatile("" ::"v"(x));
  }
  if (stop) return;  // looked at once the loads are on their way
  for (int t = n4 + (int)threadIdx.x; t < R.lds_words / 4; t += 1024)
    *(uint4 *)(w + 4 * t) = uint4{0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < NI; k++) {
    const int t = (int)threadIdx.x + 1024 * k;
    if (t < n4) *(uint4 *)(w + 4 * t) = v[k];
  }
  for (int t = (int)threadIdx.x + 1024 * NI; t < n4; t += 1024) *(uint4 *)(w + 4 * t) = img[t];
  tail_touch(desc, R.desc_bytes);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NR; k++) {
    const int t = (int)threadIdx.x + 1024 * k;
    if (t < R.rho_words) w[R.lrho0 + t] = q[k];
  }
  for (int t = (int)threadIdx.x + 1024 * NR; t < R.rho_words; t += 1024) w[R.lrho0 + t] = R.rho0[t];
  __syncthreads();
#pragma unroll 1
  for (int k = 0; k < R.nops; k++) {
    const TailOp op = ops[k];
    if (op.kind == TOP_PASS) {
      tail_pass(passes[op.pass], op.arg & TPASS_FACES, w);
      if (op.arg & TPASS_SYNC) __syncthreads();
      continue;
    }
    const TailLevel &L = tl[op.level];
    switch (op.kind) {
      case TOP_PIN: tail_pin(L, R, w); break;
      case TOP_BCPHI: tail_bc(tail_d(w, L.lphi), L.g, R); break;
      case TOP_RESREC: tail_residual_records(L, R, w); break;
      case TOP_BCRES: tail_bc(tail_d(w, L.lres), L.g, R); break;
      case TOP_RESTRICT: tail_restrict(L, tl[op.level + 1], R, w); break;
      default: tail_expand(L, tl[op.level + 1], R, w); break;
    }
  }
  const double *phi0 = tail_d(w, tl[0].lphi);
  double *out = tl[0].phi;
  TAIL_FOR(t, 2 * (int)tl[0].g.cs) { out[t] = phi0[t]; }
}
