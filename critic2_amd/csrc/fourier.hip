// Spectral derivatives of a periodic grid (grid3%fft, grid3mod@proc.f90:
// 1757-1872) and nciplot's Fourier scheme on them (nci@proc.f90:546-564), by
// transforms of the grid's lines.
//
// The reference multiplies the 3-D transform by i g (gradient), -g_c^2 or
// -|g|^2, g = sum_l b_l m_l over the indices m_l of the three axes, and takes
// the real part of the inverse.  For a real grid that real part is
//   grad_c = sum_l b_cl D_l f,
//   h_Q    = sum_l Q_ll S_l f + 2 sum_{l<m} Q_lm M_lm f
// with Q_lm = b_cl b_cm for a diagonal second derivative and sum_c b_cl b_cm
// for the Laplacian.  D_l and S_l multiply the transform along axis l alone by
// i m and -m^2.  The index range n/2-n+1..n/2 keeps an even edge's Nyquist
// term at +n/2: it is real on a real line, so i m of it is imaginary and drops
// from D, and S keeps -(n/2)^2.  M_lm = D_l D_m, and where both edges are even
// the term at both Nyquist indices, i (n_l/2) i (n_m/2), is real and stays:
// -(n_l/2)(n_m/2) P_l P_m f, P the projection on (-1)^x.
//
// So no 3-D transform is needed: a pass per axis reads a tile of lines into
// LDS, transforms it, and transforms it back twice, with i m and with -m^2,
// and the passes hand on partial sums.  What bounds it is HBM: an
// orthorhombic cell moves 76 bytes a point in three passes (grid in; gsq and
// the count of positive second derivatives out and in), any other cell 144.
// The seven complex 3-D transforms this replaces moved about 700, and their
// library plan was made anew on each call (16 ms).  Measured, whole nciplot
// calls: 256^3 orthorhombic 20.1 -> 0.57 ms (0.61 with the grid's first pass;
// kernels 143 + 201 + 251 us, 2 TB/s), 135x120x98 triclinic 19.8 -> 0.23 ms,
// 512^3 6.5 ms.  Against 80-bit sums the gradient's largest error is that of
// the 3-D transforms or less: 2e-16 to 4e-16 of the largest gradient, on
// circulant edges from 11 to 3391 1e-16 to 1.2e-15 (the 3-D transform of the
// same lines 6e-16 to 4e-15; second derivatives alike), and the error of s in
// the low-density nodes is 2 to 40 times smaller, since a line's rounding
// follows that line's values.
// Lines are transformed in pairs, packed as one complex line (both multipliers
// commute with the packing).  Edges with factors 2, 3, 5 and 7 take a
// mixed-radix Stockham transform in LDS, 8 elements a thread; other edges the
// operators' own circulant matrices, n^2 multiply-adds a line from LDS (n =
// 101: 200 a point and axis, still close to what the pass's bytes cost).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>

#include "common.hpp"
#include "nci_dev.hpp"

namespace c2 {

namespace {

constexpr int EPT = 8;          // complex elements a thread owns
constexpr int MAXT = 512;       // threads of a workgroup
// Terms of a circulant product summed before they join the total: one chain of
// n terms loses up to 5e-15 of the result on edges of 3400, sums of 64 1.1e-15.
constexpr int CIRC_SUM = 64;
// Longest line: a column tile of one pair and the constants, 3 n 16 bytes, fit
// the LDS.  Mixed radices can need more than MAXT threads before that: edges
// with a factor 5 above 2560 (n / 5 butterflies) or 3 above 3072 (n / 6).
constexpr int MAXEDGE = 3400;

// How the lines of one axis are transformed.
struct AxisPlan {
  int n;
  int dense;      // circulant matrices instead of the mixed-radix transform
  int nst;        // stages
  int rad[12];
  uint32_t mag[12];  // ceil(2^32 / Ns) of each stage: b / Ns by a multiply
  int lgw;        // 2^lgw packed line pairs a workgroup
  int tpl;        // threads of a pair; each owns the elements j, j + tpl, ...
  int threads;
};

enum { WANT_NCI = 0, WANT_GRAD = 1, WANT_HESS = 2 };

struct PassArgs {
  AxisPlan P;
  int n1, n2, n3;
  const double *f;
  int want, first, last;
  // orthorhombic: this axis's gradient scale and its Q_ll; partial sums
  double bl, ql;
  double *gsq, *h;
  int8_t *npos;
  // any cell: b[c + 3 l], the forms' Q (xx yy zz xy xz yz), D_1 f, D_2 f,
  // S_1 f and the partial second derivatives q; Nyquist projections
  double b[9];
  int nh;
  double Q[3][6];
  double *a, *bb, *s1, *q[3];
  double *c1, *c2;                      // P_1 f (y,z), P_2 f (x,z)
  const double *e12, *e13, *e23;        // P_1 P_2 f (z), P_1 P_3 f (y), P_2 P_3 f (x), or null
  // set to `call` by the first pass of a call whose grid holds a NaN or an
  // infinity, and read by its last
  unsigned long long *bad, call;
  double *out;                          // WANT_GRAD, WANT_HESS
  NciOut O;                             // WANT_NCI
};

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ __forceinline__ double2 mul_mi(double2 a) { return make_double2(a.y, -a.x); }  // -i a

// Forward transforms of R values.
template <int R>
__device__ __forceinline__ void dft(double2 *v);

template <>
__device__ __forceinline__ void dft<2>(double2 *v) {
  const double2 t = v[1];
  v[1] = csub(v[0], t);
  v[0] = cadd(v[0], t);
}
template <>
__device__ __forceinline__ void dft<4>(double2 *v) {
  const double2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]), c = cadd(v[1], v[3]), d = mul_mi(csub(v[1], v[3]));
  v[0] = cadd(a, c);
  v[1] = cadd(b, d);
  v[2] = csub(a, c);
  v[3] = csub(b, d);
}
template <>
__device__ __forceinline__ void dft<8>(double2 *v) {
  double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
  dft<4>(e);
  dft<4>(o);
  const double r = 0.70710678118654752440;
  o[1] = make_double2((o[1].x + o[1].y) * r, (o[1].y - o[1].x) * r);
  o[2] = mul_mi(o[2]);
  o[3] = make_double2((o[3].y - o[3].x) * r, -(o[3].x + o[3].y) * r);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    v[k] = cadd(e[k], o[k]);
    v[k + 4] = csub(e[k], o[k]);
  }
}
// odd R: the pairs v_j +- v_{R-j} against cos and sin of 2 pi j k / R
template <int R>
__device__ __forceinline__ void dft_odd(double2 *v, const double *c, const double *s) {
  double2 p[R / 2], m[R / 2];
  double2 sum = v[0];
#pragma unroll
  for (int j = 0; j < R / 2; j++) {
    p[j] = cadd(v[j + 1], v[R - 1 - j]);
    m[j] = csub(v[j + 1], v[R - 1 - j]);
    sum = cadd(sum, p[j]);
  }
  const double2 v0 = v[0];
  v[0] = sum;
#pragma unroll
  for (int k = 1; k <= R / 2; k++) {
    double2 re = v0, im = make_double2(0.0, 0.0);
#pragma unroll
    for (int j = 1; j <= R / 2; j++) {
      const int t = (j * k) % R;
      const double cc = c[t <= R / 2 ? t : R - t], ss = t <= R / 2 ? s[t] : -s[R - t];
      re = make_double2(re.x + cc * p[j - 1].x, re.y + cc * p[j - 1].y);
      im = make_double2(im.x + ss * m[j - 1].x, im.y + ss * m[j - 1].y);
    }
    const double2 t = mul_mi(im);
    v[k] = cadd(re, t);
    v[R - k] = csub(re, t);
  }
}
template <>
__device__ __forceinline__ void dft<3>(double2 *v) {
  const double c[2] = {1.0, -0.5}, s[2] = {0.0, 0.86602540378443864676};
  dft_odd<3>(v, c, s);
}
template <>
__device__ __forceinline__ void dft<5>(double2 *v) {
  const double c[3] = {1.0, 0.30901699437494742410, -0.80901699437494742410};
  const double s[3] = {0.0, 0.95105651629515357212, 0.58778525229247312917};
  dft_odd<5>(v, c, s);
}
template <>
__device__ __forceinline__ void dft<7>(double2 *v) {
  const double c[4] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
  const double s[4] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
  dft_odd<7>(v, c, s);
}

// Place of element k of packed line l in LDS.  Rows (AX 0) lie one after the
// other, with a gap every 8 elements against the stages' power-of-two
// strides; columns lie side by side, one element of padding per k, so that
// the last pass can read along k.
template <int AX>
__device__ __forceinline__ int lds_at(const AxisPlan &P, int k, int l) {
  return AX == 0 ? l * (P.n + P.n / 8 + 1) + k + (k >> 3) : k * ((1 << P.lgw) + 1) + l;
}

// A thread's place in the workgroup's tile: pair l, element (and butterfly)
// j, j + tpl, ... of it.  Neighbouring threads are neighbours in the grid:
// along the line in pass 0, across the lines in the others.  Threads past the
// tile own nothing.
struct Lane {
  int j, l;
};
template <int AX>
__device__ __forceinline__ Lane lane_of(const AxisPlan &P) {
  Lane t;
  const int id = (int)threadIdx.x;
  t.l = AX == 0 ? id / P.tpl : id & ((1 << P.lgw) - 1);
  t.j = AX == 0 ? id - t.l * P.tpl : id >> P.lgw;
  if (id >= P.tpl << P.lgw) {
    t.j = 1 << 24;
    t.l = 0;
  }
  return t;
}

// One Stockham stage of radix R over the whole tile, in place: all reads,
// a barrier, all writes.
template <int AX, int R>
__device__ __forceinline__ void stage(const AxisPlan &P, const Lane &t, double2 *z, const double2 *tw, int Ns,
                                      uint32_t mag) {
  constexpr int NB = EPT / R;
  const int nb = P.n / R, step = nb / Ns;
  double2 v[NB][R];
  int to[NB];
#pragma unroll
  for (int q = 0; q < NB; q++) {
    const int b = t.j + q * P.tpl;
    if (b >= nb) continue;
    const int jm = Ns == 1 ? 0 : b - (int)__umulhi((uint32_t)b, mag) * Ns;
    to[q] = (b - jm) * R + jm;
#pragma unroll
    for (int r = 0; r < R; r++) v[q][r] = z[lds_at<AX>(P, b + r * nb, t.l)];
    if (Ns > 1) {
      const double2 *w = tw;
#pragma unroll
      for (int r = 1; r < R; r++) {
        w += jm * step;
        v[q][r] = cmul(v[q][r], *w);
      }
    }
    dft<R>(v[q]);
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NB; q++) {
    if (t.j + q * P.tpl >= nb) continue;
#pragma unroll
    for (int r = 0; r < R; r++) z[lds_at<AX>(P, to[q] + r * Ns, t.l)] = v[q][r];
  }
  __syncthreads();
}

// Forward transform of the tile's packed lines (entered after a barrier).
template <int AX>
__device__ __forceinline__ void transform(const AxisPlan &P, const Lane &t, double2 *z, const double2 *tw) {
  int Ns = 1;
  for (int s = 0; s < P.nst; s++) {
    const int R = P.rad[s];
    const uint32_t mag = P.mag[s];
    switch (R) {
      case 8: stage<AX, 8>(P, t, z, tw, Ns, mag); break;
      case 7: stage<AX, 7>(P, t, z, tw, Ns, mag); break;
      case 5: stage<AX, 5>(P, t, z, tw, Ns, mag); break;
      case 4: stage<AX, 4>(P, t, z, tw, Ns, mag); break;
      case 3: stage<AX, 3>(P, t, z, tw, Ns, mag); break;
      default: stage<AX, 2>(P, t, z, tw, Ns, mag); break;
    }
    Ns *= R;
  }
}

// The axis's constants in LDS: exp(-2 pi i k/n), or the first columns of the
// circulant matrices of D (x) and S (y).  Those are taken at the distance
// q = min(k, n - k) from the diagonal, the sign of the cosine put back: sine
// and cosine of a rounded k/n near 1 would give the entries next to the
// diagonal, the largest, a relative error of n 2^-53.
__device__ __forceinline__ void load_table(const AxisPlan &P, double2 *tw) {
  for (int k = threadIdx.x; k < P.n; k += blockDim.x) {
    double s, c;
    if (P.dense) {
      const int q = 2 * k > P.n ? P.n - k : k;
      sincospi((double)q / (double)P.n, &s, &c);
      c = q < k ? -c : c;
      const double sg = (k & 1) ? -0.5 : 0.5, n = P.n;
      if (k == 0)
        tw[k] = make_double2(0.0, -(P.n & 1 ? n * n - 1.0 : n * n + 2.0) / 12.0);
      else
        tw[k] = make_double2(P.n & 1 ? sg / s : sg * c / s, -2.0 * sg * 0.5 * (P.n & 1 ? c : 1.0) / (s * s));
    } else {
      sincospi(-2.0 * (double)k / (double)P.n, &s, &c);
      tw[k] = make_double2(c, s);
    }
  }
}

// D and S of the workgroup's lines on a circulant edge: IB neighbouring outputs
// of a line at a time; the matrices' entries slide through registers as j
// advances.  S: also the second derivatives.
template <int AX, bool S>
__device__ __forceinline__ void circulant(const AxisPlan &P, const Lane &t, double2 *z, const double2 *tw,
                                          double2 d[EPT], double2 s[EPT], double2 *nyq) {
  constexpr int IB = 4, NU = EPT / IB, STEP = 8;  // STEP: w is back in place after it
  double2 od[NU][IB], os[NU][IB];
#pragma unroll
  for (int u = 0; u < NU; u++) {
    const int i0 = (t.j + u * P.tpl) * IB;
    if (i0 >= P.n) continue;
    double2 w[IB], pd[IB] = {}, ps[IB] = {};
#pragma unroll
    for (int r = 0; r < IB; r++) {
      od[u][r] = os[u][r] = make_double2(0.0, 0.0);
      w[r] = tw[(i0 + r) % P.n];
    }
    int nx = i0;  // index of w[0]
    double2 ny = make_double2(0.0, 0.0);
    auto term = [&](int j) {
      const double2 v = z[lds_at<AX>(P, j, t.l)];
#pragma unroll
      for (int r = 0; r < IB; r++) {
        pd[r] = make_double2(pd[r].x + w[r].x * v.x, pd[r].y + w[r].x * v.y);
        if (S) ps[r] = make_double2(ps[r].x + w[r].y * v.x, ps[r].y + w[r].y * v.y);
      }
      if (nyq && i0 == 0) ny = (j & 1) ? csub(ny, v) : cadd(ny, v);
      nx = nx == 0 ? P.n - 1 : nx - 1;
#pragma unroll
      for (int r = IB - 1; r > 0; r--) w[r] = w[r - 1];
      w[0] = tw[nx];
    };
    auto total = [&]() {
#pragma unroll
      for (int r = 0; r < IB; r++) {
        od[u][r] = cadd(od[u][r], pd[r]);
        os[u][r] = cadd(os[u][r], ps[r]);
        pd[r] = ps[r] = make_double2(0.0, 0.0);
      }
    };
    int j = 0;
    for (; j + STEP <= P.n; j += STEP) {
#pragma unroll
      for (int e = 0; e < STEP; e++) term(j + e);
      if ((j + STEP) % CIRC_SUM == 0) total();
    }
    for (; j < P.n; j++) term(j);
    total();
    if (nyq && i0 == 0) nyq[t.l] = cscale(ny, 1.0 / (double)P.n);
  }
#pragma unroll
  for (int pass = 0; pass < (S ? 2 : 1); pass++) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NU; u++) {
      const int i0 = (t.j + u * P.tpl) * IB;
#pragma unroll
      for (int r = 0; r < IB; r++)
        if (i0 + r < P.n) z[lds_at<AX>(P, i0 + r, t.l)] = pass == 0 ? od[u][r] : os[u][r];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < EPT; q++) {
      const int k = t.j + q * P.tpl;
      if (k >= P.n) continue;
      (pass == 0 ? d : s)[q] = z[lds_at<AX>(P, k, t.l)];
    }
  }
}

// D and S of the workgroup's lines: x[q] are this thread's elements, and so
// are d[q] and s[q] (s only if wants).  nyq, when not null, receives the
// lines' P values (the transform at n/2 over n; n even), one packed pair per
// line.
template <int AX>
__device__ __forceinline__ void derivatives(const AxisPlan &P, const Lane &t, double2 *z, const double2 *tw,
                                            const double2 x[EPT], bool wants, double2 d[EPT], double2 s[EPT],
                                            double2 *nyq) {
  const double rn = 1.0 / (double)P.n;
#pragma unroll
  for (int q = 0; q < EPT; q++) {
    const int k = t.j + q * P.tpl;
    if (k < P.n) z[lds_at<AX>(P, k, t.l)] = x[q];
  }
  __syncthreads();
  if (!P.dense) {
    transform<AX>(P, t, z, tw);
    double2 K[EPT];
#pragma unroll
    for (int q = 0; q < EPT; q++) {
      const int k = t.j + q * P.tpl;
      if (k >= P.n) continue;
      double2 &w = z[lds_at<AX>(P, k, t.l)];
      K[q] = cscale(w, rn);
      if (nyq && 2 * k == P.n) nyq[t.l] = K[q];
      // i m K with its parts swapped: the forward transform of a swapped
      // value is the swapped inverse
      const double m = 2 * k == P.n ? 0.0 : (double)(2 * k > P.n ? k - P.n : k);
      w = make_double2(m * K[q].x, -m * K[q].y);
    }
    __syncthreads();
    transform<AX>(P, t, z, tw);
#pragma unroll
    for (int q = 0; q < EPT; q++) {
      const int k = t.j + q * P.tpl;
      if (k >= P.n) continue;
      double2 &w = z[lds_at<AX>(P, k, t.l)];
      d[q] = make_double2(w.y, w.x);
      const double m = (double)(2 * k > P.n ? k - P.n : k);
      w = make_double2(-m * m * K[q].y, -m * m * K[q].x);
    }
    if (!wants) return;
    __syncthreads();
    transform<AX>(P, t, z, tw);
#pragma unroll
    for (int q = 0; q < EPT; q++) {
      const int k = t.j + q * P.tpl;
      if (k >= P.n) continue;
      const double2 w = z[lds_at<AX>(P, k, t.l)];
      s[q] = make_double2(w.y, w.x);
    }
    return;
  }
  if (wants)
    circulant<AX, true>(P, t, z, tw, d, s, nyq);
  else
    circulant<AX, false>(P, t, z, tw, d, s, nyq);
}

// Where the thread's pair of lines lies in the grid: element k at p + k st,
// the second line's at that + second; v0, v1: the lines exist.
struct Place {
  int64_t p, st, second;
  bool v0, v1;
};
template <int AX>
__device__ __forceinline__ Place place_of(const PassArgs &A, int tile, int group, const Lane &t) {
  Place g;
  if (AX == 0) {
    const int64_t rows = (int64_t)A.n2 * A.n3, r = 2 * (((int64_t)tile << A.P.lgw) + t.l);
    g.v0 = r < rows;
    g.v1 = r + 1 < rows;
    g.p = r * A.n1;
    g.st = 1;
    g.second = A.n1;
  } else {
    const int x = 2 * ((tile << A.P.lgw) + t.l);
    g.v0 = x < A.n1;
    g.v1 = x + 1 < A.n1;
    g.p = (int64_t)x + (int64_t)A.n1 * (AX == 1 ? (int64_t)A.n2 * group : (int64_t)group);
    g.st = AX == 1 ? A.n1 : (int64_t)A.n1 * A.n2;
    g.second = 1;
  }
  return g;
}
__device__ __forceinline__ double2 ld2(const double *p, const Place &g, int64_t o) {
  return make_double2(g.v0 ? p[o] : 0.0, g.v1 ? p[o + g.second] : 0.0);
}
__device__ __forceinline__ void st2(double *p, const Place &g, int64_t o, double2 v) {
  if (g.v0) p[o] = v.x;
  if (g.v1) p[o + g.second] = v.y;
}
// The thread's elements of a grid.
__device__ __forceinline__ void load_tile(const AxisPlan &P, const Lane &t, const Place &g, const double *p,
                                          double2 v[EPT]) {
#pragma unroll
  for (int q = 0; q < EPT; q++) {
    const int k = t.j + q * P.tpl;
    v[q] = make_double2(0.0, 0.0);
    if (k < P.n) v[q] = ld2(p, g, g.p + k * g.st);
  }
}

// A NaN or an infinity anywhere in the grid makes every derivative NaN, as it
// does in the reference's 3-D transform, though a line transform carries it to
// its own lines only: the first pass, which transforms every line, notes it
// from each thread's first derivative, NaN or infinite with any of its line.
__device__ __forceinline__ void note_nonfinite(const PassArgs &A, double2 d) {
  if (!__builtin_isfinite(d.x) || !__builtin_isfinite(d.y))
    __hip_atomic_store(A.bad, A.call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// nci@proc.f90:598-599: crho and s of a node; npos positive diagonal second
// derivatives (nci@proc.f90:546-564)
__device__ __forceinline__ void nci_value(double f, double gsq, int npos, double &crho, double &s) {
  const double cst = 6.18733545256027186;  // 2 (3 pi^2)^(1/3)
  const double den = f > 1e-80 ? f : 1e-80;
  s = sqrt(gsq) / (cst * (den * cbrt(den)));
  const double a = fabs(f) * 100.0;
  crho = npos >= 2 ? a : -a;
}

// The finished node values of the last pass, written in the outputs' order.
// AX 2 with z fastest goes through LDS so that neighbouring lanes write
// neighbouring k.
template <int AX>
__device__ __forceinline__ void store_nci(const PassArgs &A, int tile, int group, const Lane &t, const Place &g,
                                          double2 *z, const double2 cr[EPT], const double2 sv[EPT]) {
  const AxisPlan &P = A.P;
  double *oc = (double *)A.O.crho, *os = (double *)A.O.cgrad;
  if (AX == 2 && A.O.zfast) {
    const int lw2 = 2 << P.lgw, pitch = lw2 + 2;
    const double *zs = reinterpret_cast<const double *>(z);
#pragma unroll
    for (int which = 0; which < 2; which++) {
      __syncthreads();
#pragma unroll
      for (int q = 0; q < EPT; q++) {
        const int k = t.j + q * P.tpl;
        if (k < P.n) z[lds_at<AX>(P, k, t.l)] = which ? sv[q] : cr[q];
      }
      __syncthreads();
      double *o = which ? os : oc;
      // a wavefront takes a column at a time
      for (int c = threadIdx.x >> 6; c < lw2; c += blockDim.x >> 6) {
        const int x = tile * lw2 + c;
        if (x >= A.n1) break;
        double *oo = o + (size_t)A.n3 * ((size_t)group + (size_t)A.n2 * x);
        for (int k = threadIdx.x & 63; k < P.n; k += 64) oo[k] = zs[k * pitch + c];
      }
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < EPT; q++) {
    const int k = t.j + q * P.tpl;
    if (k >= P.n) continue;
    st2(oc, g, g.p + k * g.st, cr[q]);
    st2(os, g, g.p + k * g.st, sv[q]);
  }
}

// One axis of an orthorhombic cell: b has one Cartesian component per axis, so
// |grad f|^2 is the sum of the axes' (b_l D_l f)^2 and a diagonal second
// derivative is one axis's.
template <int AX>
__global__ void __launch_bounds__(MAXT) k_line_ortho(PassArgs A) {
  extern __shared__ double2 lds[];
  const AxisPlan &P = A.P;
  double2 *tw = lds, *z = lds + P.n;
  const int tiles = AX == 0 ? 1 : (A.n1 + (2 << P.lgw) - 1) / (2 << P.lgw);  // of a group
  const int group = AX == 0 ? 0 : blockIdx.x / tiles, tile = blockIdx.x - (AX == 0 ? 0 : group * tiles);
  const Lane t = lane_of<AX>(P);
  const Place g = place_of<AX>(A, tile, group, t);
  double2 x[EPT], d[EPT], s[EPT];
  load_tile(P, t, g, A.f, x);
  load_table(P, tw);
#pragma unroll
  for (int q = 0; q < EPT; q++) d[q] = s[q] = make_double2(0.0, 0.0);
  derivatives<AX>(P, t, z, tw, x, A.want != WANT_GRAD, d, s, nullptr);
  if (A.first) note_nonfinite(A, d[0]);
  const bool bad = A.last && !A.first && *A.bad == A.call;
  const double nan = __builtin_nan("");
#pragma unroll
  for (int q = 0; q < EPT; q++) {
    const int k = t.j + q * P.tpl;
    if (k >= P.n) continue;
    const int64_t o = g.p + k * g.st;
    if (A.want == WANT_HESS) {
      double2 h = cscale(s[q], A.ql);
      if (!A.first) h = cadd(h, ld2(A.h, g, o));
      if (bad) h = make_double2(nan, nan);
      st2(A.last ? A.out : A.h, g, o, h);
      continue;
    }
    const double gx = A.bl * d[q].x, gy = A.bl * d[q].y;
    double2 gs = make_double2(gx * gx, gy * gy);
    if (!A.first) gs = cadd(gs, ld2(A.gsq, g, o));
    if (bad) gs = make_double2(nan, nan);
    if (A.want == WANT_GRAD) {
      if (A.last)
        st2(A.out, g, o, make_double2(sqrt(gs.x), sqrt(gs.y)));
      else
        st2(A.gsq, g, o, gs);
      continue;
    }
    int c0 = s[q].x > 0.0, c1 = s[q].y > 0.0;
    if (!A.first) {
      if (g.v0) c0 += A.npos[o];
      if (g.v1) c1 += A.npos[o + g.second];
    }
    if (!A.last) {
      st2(A.gsq, g, o, gs);
      if (g.v0) A.npos[o] = (int8_t)c0;
      if (g.v1) A.npos[o + g.second] = (int8_t)c1;
    } else {
      const double2 f = ld2(A.f, g, o);  // again: not held through the transforms
      nci_value(f.x, gs.x, bad ? 0 : c0, d[q].x, s[q].x);
      nci_value(f.y, gs.y, bad ? 0 : c1, d[q].y, s[q].y);
    }
  }
  if (A.last && A.want == WANT_NCI) store_nci<AX>(A, tile, group, t, g, z, d, s);
}

// One axis of any cell, in the order 0, 1, 2.  Pass 0 leaves D_1 f and S_1 f,
// pass 1 D_2 f and the forms over axes 1 and 2, pass 2 finishes.
template <int AX>
__global__ void __launch_bounds__(MAXT) k_line_any(PassArgs A) {
  extern __shared__ double2 lds[];
  const AxisPlan &P = A.P;
  double2 *tw = lds, *z = lds + P.n;
  const int tiles = AX == 0 ? 1 : (A.n1 + (2 << P.lgw) - 1) / (2 << P.lgw);
  const int group = AX == 0 ? 0 : blockIdx.x / tiles, tile = blockIdx.x - (AX == 0 ? 0 : group * tiles);
  const bool hess = A.want != WANT_GRAD;
  __shared__ double2 nyq[8];
  const Lane t = lane_of<AX>(P);
  const Place g = place_of<AX>(A, tile, group, t);
  load_table(P, tw);
  double2 x[EPT], d[EPT], s[EPT], m1[EPT], m2[EPT], none[EPT];
#pragma unroll
  for (int q = 0; q < EPT; q++) d[q] = s[q] = m1[q] = m2[q] = make_double2(0.0, 0.0);
  if (AX == 2 && hess) {  // M_13 and M_23 first: the rest is then read once, at the end
    load_tile(P, t, g, A.a, x);
    derivatives<AX>(P, t, z, tw, x, false, m1, none, nullptr);
    load_tile(P, t, g, A.bb, x);
    derivatives<AX>(P, t, z, tw, x, false, m2, none, nullptr);
  }
  load_tile(P, t, g, A.f, x);
  double *cn = AX == 0 ? A.c1 : AX == 1 ? A.c2 : nullptr;
  derivatives<AX>(P, t, z, tw, x, hess, d, s, cn ? nyq : nullptr);
  if (AX == 0) note_nonfinite(A, d[0]);
  const bool bad = AX == 2 && *A.bad == A.call;
  const double nan = __builtin_nan("");
  if (cn) {  // the packed lines' Nyquist projections, by each pair's first thread
    __syncthreads();
    if (t.j == 0) {
      const int64_t o = AX == 0 ? 2 * (((int64_t)tile << P.lgw) + t.l)
                                : 2 * ((tile << P.lgw) + t.l) + (int64_t)A.n1 * group;
      if (g.v0) cn[o] = nyq[t.l].x;
      if (g.v1) cn[o + 1] = nyq[t.l].y;
    }
  }
  if (AX == 1 && hess) {
    load_tile(P, t, g, A.a, x);
    derivatives<AX>(P, t, z, tw, x, false, m1, none, nullptr);
  }
  // M's terms at two Nyquist indices; a pair's first column is even in P_1
  const double e12 = AX == 1 && A.e12 ? -0.25 * A.n1 * A.n2 * A.e12[group] : 0.0;
  const double e13 = AX == 2 && A.e13 ? -0.25 * A.n1 * A.n3 * A.e13[group] : 0.0;
  double2 e23 = make_double2(0.0, 0.0);
  if (AX == 2 && A.e23) {
    const int col = 2 * ((tile << P.lgw) + t.l);
    const double sg = (group & 1) ? 0.25 * A.n2 * A.n3 : -0.25 * A.n2 * A.n3;
    e23 = make_double2(g.v0 ? sg * A.e23[col] : 0.0, g.v1 ? sg * A.e23[col + 1] : 0.0);
  }
#pragma unroll
  for (int q = 0; q < EPT; q++) {
    const int k = t.j + q * P.tpl;
    if (k >= P.n) continue;
    const int64_t o = g.p + k * g.st;
    const double sg = (k & 1) ? -1.0 : 1.0;
    if (AX == 0) {
      st2(A.a, g, o, d[q]);
      if (hess) st2(A.s1, g, o, s[q]);
      continue;
    }
    if (AX == 1) {
      st2(A.bb, g, o, d[q]);
      if (!hess) continue;
      const double2 m = make_double2(m1[q].x + sg * e12, m1[q].y - sg * e12), u = ld2(A.s1, g, o);
#pragma unroll
      for (int w = 0; w < 3; w++)
        if (w < A.nh)
          st2(A.q[w], g, o, make_double2(A.Q[w][0] * u.x + A.Q[w][1] * s[q].x + 2.0 * A.Q[w][3] * m.x,
                                         A.Q[w][0] * u.y + A.Q[w][1] * s[q].y + 2.0 * A.Q[w][3] * m.y));
      continue;
    }
    double2 h[3] = {};
    if (hess) {
      const double2 a = make_double2(m1[q].x + sg * e13, m1[q].y - sg * e13);
      const double2 b = make_double2(m2[q].x + sg * e23.x, m2[q].y + sg * e23.y);
#pragma unroll
      for (int w = 0; w < 3; w++)
        if (w < A.nh) {
          const double2 u = ld2(A.q[w], g, o);
          h[w].x = u.x + A.Q[w][2] * s[q].x + 2.0 * (A.Q[w][4] * a.x + A.Q[w][5] * b.x);
          h[w].y = u.y + A.Q[w][2] * s[q].y + 2.0 * (A.Q[w][4] * a.y + A.Q[w][5] * b.y);
        }
    }
    if (bad) h[0] = h[1] = h[2] = make_double2(nan, nan);
    if (A.want == WANT_HESS) {
      st2(A.out, g, o, h[0]);
      continue;
    }
    const double2 da = ld2(A.a, g, o), db = ld2(A.bb, g, o);
    double2 gs = make_double2(0.0, 0.0);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double gx = A.b[c] * da.x + A.b[c + 3] * db.x + A.b[c + 6] * d[q].x;
      const double gy = A.b[c] * da.y + A.b[c + 3] * db.y + A.b[c + 6] * d[q].y;
      gs = make_double2(gs.x + gx * gx, gs.y + gy * gy);
    }
    if (bad) gs = make_double2(nan, nan);
    if (A.want == WANT_GRAD) {
      st2(A.out, g, o, make_double2(sqrt(gs.x), sqrt(gs.y)));
      continue;
    }
    const double2 f = ld2(A.f, g, o);
    nci_value(f.x, gs.x, (h[0].x > 0.0) + (h[1].x > 0.0) + (h[2].x > 0.0), d[q].x, s[q].x);
    nci_value(f.y, gs.y, (h[0].y > 0.0) + (h[1].y > 0.0) + (h[2].y > 0.0), d[q].y, s[q].y);
  }
  if (AX == 2 && A.want == WANT_NCI) store_nci<AX>(A, tile, group, t, g, z, d, s);
}

// A call of one pass: its derivatives made NaN where the pass noted a NaN or
// an infinity.
__global__ void __launch_bounds__(256) k_line_nan(const unsigned long long *bad, unsigned long long call, uint64_t n,
                                                  double *out) {
  if (*bad != call) return;
  for (uint64_t p = (uint64_t)blockIdx.x * 256 + threadIdx.x; p < n; p += (uint64_t)gridDim.x * 256)
    out[p] = __builtin_nan("");
}

// out[o] = (1/n) sum_q (-1)^q in[o so + q sq]: one wavefront each
__global__ void __launch_bounds__(64) k_alternating(const double *in, int64_t so, int64_t sq, int n, double *out) {
  double v = 0.0;
  for (int q = threadIdx.x; q < n; q += 64) {
    const double t = in[(int64_t)blockIdx.x * so + (int64_t)q * sq];
    v += (q & 1) ? -t : t;
  }
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  if (threadIdx.x == 0) out[blockIdx.x] = v / (double)n;
}

// Radices of n (8 first: fewest stages), or dense; line pairs and threads of
// a workgroup.  8 pairs make the column passes' reads whole 128-byte lines;
// long lines take fewer so that 512 threads own the tile.
AxisPlan make_axis(int n) {
  AxisPlan P{};
  P.n = n;
  int m = n;
  for (int r : {8, 7, 5, 4, 3, 2})
    while (m % r == 0 && P.nst < 12) {
      P.rad[P.nst++] = r;
      m /= r;
    }
  P.dense = m != 1;
  if (P.dense) P.nst = 0;
  uint32_t Ns = 1;
  // every element, butterfly and block of outputs must be some thread's
  int need = (n + EPT - 1) / EPT;
  for (int s = 0; s < P.nst; s++) {
    const int nb = EPT / P.rad[s], t = (n / P.rad[s] + nb - 1) / nb;
    need = t > need ? t : need;
    P.mag[s] = Ns == 1 ? 0u : (uint32_t)(((1ull << 32) + Ns - 1) / Ns);
    Ns *= P.rad[s];
  }
  P.tpl = (need + 7) / 8 * 8;
  for (P.lgw = 3; P.lgw > 0 && P.tpl << P.lgw > MAXT;) P.lgw--;
  P.threads = (P.tpl << P.lgw) <= MAXT ? ((P.tpl << P.lgw) + 63) / 64 * 64 : 0;
  return P;
}

size_t lds_bytes(const AxisPlan &P, int ax) {
  const size_t lw = (size_t)1 << P.lgw;
  const size_t z = ax == 0 ? lw * (P.n + P.n / 8 + 1) : (size_t)P.n * (lw + 1);
  return sizeof(double2) * (z + P.n);
}

template <class K>
void launch_pass(c2gpu_ctx *ctx, const char *name, K kern, int ax, PassArgs &A) {
  const int64_t per = 2ll << A.P.lgw;
  const int64_t rows = (int64_t)A.n2 * A.n3;
  const int64_t nblk = ax == 0 ? (rows + per - 1) / per : (A.n1 + per - 1) / per * (ax == 1 ? A.n3 : A.n2);
  const size_t lds = lds_bytes(A.P, ax);
  C2_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)lds));
  (void)grid_for(nblk * A.P.threads, A.P.threads);  // refuses more than one dispatch holds
  hipEvent_t a = nullptr, b = nullptr;
  if (ctx->timing) {
    a = event_get(ctx);
    b = event_get(ctx);
    C2_HIP(hipEventRecord(a, ctx->stream));
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(A.P.threads), lds, ctx->stream, A);
  C2_HIP(hipGetLastError());
  if (ctx->timing) {
    C2_HIP(hipEventRecord(b, ctx->stream));
    ctx->pending.push_back({name, a, b});
  }
}

}  // namespace

// Whether the line passes take a grid with these edges: none above MAXEDGE, and
// none whose butterflies need more than MAXT threads.
bool fourier_lines_ok(const int n[3]) {
  for (int a = 0; a < 3; a++)
    if (n[a] > MAXEDGE || make_axis(n[a]).threads == 0) return false;
  return true;
}

// The derivative grid `kind` (C2GPU_FT_*) of the device grid f into out, or,
// with kind < 0, nciplot's crho and cgrad into O (FP64).  bvec: reciprocal
// vectors, column l that of axis l, scaled by 2 pi.
void fourier_lines_run(c2gpu_ctx *ctx, const double *f, const int n[3], const double bvec[9], int kind, double *out,
                       const NciOut *O) {
  const size_t N = (size_t)n[0] * n[1] * n[2];
  PassArgs A{};
  A.n1 = n[0];
  A.n2 = n[1];
  A.n3 = n[2];
  A.f = f;
  A.out = out;
  A.want = kind < 0 ? WANT_NCI : kind == C2GPU_FT_GRAD ? WANT_GRAD : WANT_HESS;
  if (O) A.O = *O;
  // the quadratic forms wanted
  A.nh = A.want == WANT_NCI ? 3 : A.want == WANT_HESS ? 1 : 0;
  for (int w = 0; w < A.nh; w++) {
    const int pr[6][2] = {{0, 0}, {1, 1}, {2, 2}, {0, 1}, {0, 2}, {1, 2}};
    for (int t = 0; t < 6; t++)
      for (int c = 0; c < 3; c++) {
        const bool in = A.want == WANT_NCI ? c == w : kind == C2GPU_FT_LAP || c == kind - C2GPU_FT_XX;
        if (in) A.Q[w][t] += bvec[c + 3 * pr[t][0]] * bvec[c + 3 * pr[t][1]];
      }
  }
  std::memcpy(A.b, bvec, sizeof A.b);
  // calls are numbered, so the word is cleared once, not before each call
  A.bad = buf<unsigned long long>(ctx, "fourier_bad", 1);
  if (ctx->fourier_calls == 0) C2_HIP(hipMemsetAsync(A.bad, 0, sizeof *A.bad, ctx->stream));
  A.call = ++ctx->fourier_calls;
  // Orthorhombic: one Cartesian component per axis, a different one each.
  // Components below 1e-15 of the largest (a right angle's cosine is 6e-17)
  // change the derivatives by less than the transforms' own rounding.
  double big = 0.0;
  for (int q = 0; q < 9; q++) big = std::fmax(big, std::fabs(bvec[q]));
  int comp[3], used = 0;
  bool ortho = true;
  for (int l = 0; l < 3; l++) {
    int cnt = 0;
    for (int c = 0; c < 3; c++)
      if (std::fabs(bvec[c + 3 * l]) > 1e-15 * big) {
        comp[l] = c;
        cnt++;
        used |= 1 << c;
      }
    ortho = ortho && cnt == 1;
  }
  ortho = ortho && used == 7;
  const AxisPlan plan[3] = {make_axis(n[0]), make_axis(n[1]), make_axis(n[2])};
  if (ortho) {
    int list[3], m = 0;
    for (int l = 0; l < 3; l++)
      if (A.want != WANT_HESS || kind == C2GPU_FT_LAP || comp[l] == kind - C2GPU_FT_XX) list[m++] = l;
    if (A.want == WANT_HESS && m > 1) A.h = buf<double>(ctx, "fourier_h", N);
    if (A.want != WANT_HESS) A.gsq = buf<double>(ctx, "fourier_gsq", N);
    if (A.want == WANT_NCI) A.npos = buf<int8_t>(ctx, "fourier_npos", N);
    for (int p = 0; p < m; p++) {
      const int l = list[p];
      A.P = plan[l];
      A.first = p == 0;
      A.last = p == m - 1;
      A.bl = bvec[comp[l] + 3 * l];
      A.ql = A.bl * A.bl;
      if (l == 0)
        launch_pass(ctx, "k_line_ortho<0>", k_line_ortho<0>, 0, A);
      else if (l == 1)
        launch_pass(ctx, "k_line_ortho<1>", k_line_ortho<1>, 1, A);
      else
        launch_pass(ctx, "k_line_ortho<2>", k_line_ortho<2>, 2, A);
    }
    if (m == 1)
      C2_LAUNCH(ctx, k_line_nan, dim3((unsigned)std::min<size_t>((N + 255) / 256, 2048)), dim3(256), 0,
                (const unsigned long long *)A.bad, A.call, (uint64_t)N, out);
    return;
  }
  A.a = buf<double>(ctx, "fourier_gsq", N);
  A.bb = buf<double>(ctx, "fourier_h", N);
  double *e12 = nullptr, *e13 = nullptr, *e23 = nullptr;
  if (A.nh) {
    A.s1 = buf<double>(ctx, "fourier_s", N);
    for (int w = 0; w < A.nh; w++) A.q[w] = buf<double>(ctx, "fourier_q" + std::to_string(w), N);
    const bool ev1 = n[0] % 2 == 0, ev2 = n[1] % 2 == 0, ev3 = n[2] % 2 == 0;
    if (ev1 && (ev2 || ev3)) A.c1 = buf<double>(ctx, "fourier_c1", (size_t)n[1] * n[2]);
    if (ev2 && ev3) A.c2 = buf<double>(ctx, "fourier_c2", (size_t)n[0] * n[2]);
    if (ev1 && ev2) e12 = buf<double>(ctx, "fourier_e12", n[2]);
    if (ev1 && ev3) e13 = buf<double>(ctx, "fourier_e13", n[1]);
    if (ev2 && ev3) e23 = buf<double>(ctx, "fourier_e23", n[0]);
  }
  A.P = plan[0];
  launch_pass(ctx, "k_line_any<0>", k_line_any<0>, 0, A);
  // c1(y,z): P_1 f; its alternating sums over y and over z
  if (e12) C2_LAUNCH(ctx, k_alternating, dim3(n[2]), dim3(64), 0, (const double *)A.c1, (int64_t)n[1], (int64_t)1, n[1], e12);
  if (e13) C2_LAUNCH(ctx, k_alternating, dim3(n[1]), dim3(64), 0, (const double *)A.c1, (int64_t)1, (int64_t)n[1], n[2], e13);
  A.e12 = e12;
  A.P = plan[1];
  launch_pass(ctx, "k_line_any<1>", k_line_any<1>, 1, A);
  if (e23) C2_LAUNCH(ctx, k_alternating, dim3(n[0]), dim3(64), 0, (const double *)A.c2, (int64_t)1, (int64_t)n[0], n[2], e23);
  A.e13 = e13;
  A.e23 = e23;
  A.P = plan[2];
  launch_pass(ctx, "k_line_any<2>", k_line_any<2>, 2, A);
}

}  // namespace c2
