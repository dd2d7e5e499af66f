// Device definitions shared by the NCI sources: the bricks of 256 nodes, the
// output layout of nciplot's crho/cgrad arrays (nci@proc.f90:502-505) and the
// middle eigenvalue of the Hessian.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace c2 {

static const double PI_D = 3.14159265358979323846264338327950288;

// The nodes: those of a periodic grid of the cell x2c (box == 0), at
// x2c (i/n1, j/n2, k/n3), or those of an nciplot cube (box == 1), at
// x0 + i xm(:,1) + j xm(:,2) + k xm(:,3) (nci@proc.f90:548).
struct Geo {
  int n1, n2, n3;
  // bricks of 256 nodes: 2^lx x 2^ly x 2^lz, nb per axis; zf: threads and
  // bricks run z fastest, for kernels whose outputs do (else x fastest)
  int nb1, nb2, nb3;
  int lx, ly, lz, zf;
  double x2c[9];
  int box;
  double x0[3], xm[9];
};

// Cartesian position at real-valued node coordinates (u, v, w).
__device__ __forceinline__ void geo_cart(const Geo &G, double u, double v, double w, double xc[3]) {
  if (G.box) {
#pragma unroll
    for (int r = 0; r < 3; r++) xc[r] = G.x0[r] + u * G.xm[r] + v * G.xm[r + 3] + w * G.xm[r + 6];
  } else {
    const double f0 = u / G.n1, f1 = v / G.n2, f2 = w / G.n3;
#pragma unroll
    for (int r = 0; r < 3; r++) xc[r] = G.x2c[r] * f0 + G.x2c[r + 3] * f1 + G.x2c[r + 6] * f2;
  }
}

__device__ __forceinline__ void node_cart(const Geo &G, int i, int j, int k, double xc[3]) {
  geo_cart(G, (double)i, (double)j, (double)k, xc);
}

// Node (0, 0, 0) of brick b.
__device__ __forceinline__ void brick_origin(const Geo &G, int b, int &i, int &j, int &k) {
  const int na = G.zf ? G.nb3 : G.nb1;
  const int r = b / na, a = b - r * na;
  const int b2 = r % G.nb2, c = r / G.nb2;
  i = (G.zf ? c : a) << G.lx;
  j = b2 << G.ly;
  k = (G.zf ? a : c) << G.lz;
}
// Node of thread t (of 256) of brick b; false when it lies past the grid.
__device__ __forceinline__ bool brick_node(const Geo &G, int b, int t, int &i, int &j, int &k) {
  brick_origin(G, b, i, j, k);
  const int la = G.zf ? G.lz : G.lx;
  const int a = t & ((1 << la) - 1), u = t >> la, y = u & ((1 << G.ly) - 1), c = u >> G.ly;
  i += G.zf ? c : a;
  j += y;
  k += G.zf ? a : c;
  return i < G.n1 && j < G.n2 && k < G.n3;
}
// Cartesian middle of brick b's nodes.
__device__ __forceinline__ void brick_middle(const Geo &G, int b, double c[3]) {
  int i, j, k;
  brick_origin(G, b, i, j, k);
  geo_cart(G, i + 0.5 * ((1 << G.lx) - 1), j + 0.5 * ((1 << G.ly) - 1), k + 0.5 * ((1 << G.lz) - 1), c);
}

// Middle eigenvalue of a symmetric 3x3 matrix (trigonometric closed form of
// the characteristic cubic).
template <class T>
__device__ inline T eig_mid_t(T h00, T h11, T h22, T h01, T h02, T h12) {
  const T p1 = h01 * h01 + h02 * h02 + h12 * h12;
  if (p1 == T(0)) {  // diagonal
    T a = h00, b = h11, c = h22, t;
    if (a > b) { t = a; a = b; b = t; }
    if (b > c) { t = b; b = c; c = t; }
    if (a > b) { t = a; a = b; b = t; }
    return b;
  }
  const T q = (h00 + h11 + h22) / T(3);
  const T d0 = h00 - q, d1 = h11 - q, d2 = h22 - q;
  const T p2 = d0 * d0 + d1 * d1 + d2 * d2 + T(2) * p1;
  const T p = sqrt(p2 / T(6));
  const T ip = T(1) / p;
  const T b00 = d0 * ip, b11 = d1 * ip, b22 = d2 * ip, b01 = h01 * ip, b02 = h02 * ip, b12 = h12 * ip;
  T detb = b00 * (b11 * b22 - b12 * b12) - b01 * (b01 * b22 - b12 * b02) + b02 * (b01 * b12 - b11 * b02);
  T rr = detb / T(2);
  rr = rr < T(-1) ? T(-1) : (rr > T(1) ? T(1) : rr);
  const T phi = acos(rr) / T(3);
  const T l1 = q + T(2) * p * cos(phi);
  const T l3 = q + T(2) * p * cos(phi + T(2.0943951023931954923));
  return T(3) * q - l1 - l3;
}

// Whether eig_mid_t's middle eigenvalue is negative (a negative zero too).
// All eigenvalues are real, so the signs of the determinant d, the trace t and
// the sum m of the principal minors settle how many are negative.  That is
// taken where the middle eigenvalue l is surely further from zero than either
// way's rounding: |l| <= x F implies |d| <= x F (|m| + sqrt(2) x F^2), F the
// Frobenius norm, since d = l (m - l (l1 + l3)).  x = 2e-3 is eight times the
// closed form's FP32 error, largest (2.3e-4 F) at a double eigenvalue, where
// acos is flat.  Elsewhere, and for zeros, infinities and NaN, the closed form
// decides, so the answer is its own wherever it loses no squares: entries below
// 1e18 and a traceless part above 1e-18 in FP32, 1e152 and 1e-152 in FP64.  Past
// that, where no density table in use reaches, the signs settled here are the
// right ones and the closed form's need not be.  About 45 operations instead of
// an acos and two cosines.
template <class T>
__device__ __forceinline__ bool eig_mid_negative(T h00, T h11, T h22, T h01, T h02, T h12) {
  T mx = fmax(fmax(fmax(fabs(h00), fabs(h11)), fmax(fabs(h22), fabs(h01))), fmax(fabs(h02), fabs(h12)));
  const T sc = sizeof(T) == 4 ? (T)__builtin_amdgcn_rcpf((float)mx) : (T)__builtin_amdgcn_rcp((double)mx);
  const T a = h00 * sc, b = h11 * sc, c = h22 * sc, u = h01 * sc, v = h02 * sc, w = h12 * sc;
  const T off = u * u + v * v + w * w;
  const T t = a + b + c, m = a * b + a * c + b * c - off;
  const T d = a * (b * c - w * w) - u * (u * c - w * v) + v * (u * w - b * v);
  const T f2 = a * a + b * b + c * c + T(2) * off;
  const T x = T(2e-3);
  const T lim = x * (fabs(m) + T(1.5) * x * f2);
  if (d * d > lim * lim * f2) return d > T(0) ? !(t > T(0) && m > T(0)) : (t < T(0) && m > T(0));
  const T l2 = eig_mid_t<T>(h00, h11, h22, h01, h02, h12);
  return l2 < T(0) || (l2 == T(0) && signbit(l2));
}

struct NciOut {
  void *crho, *cgrad;  // double* or float*
  int is_f32;
  int zfast;
  void *rhoat = nullptr;  // promolecular density (same type), when wanted
};

__device__ __forceinline__ size_t out_index(const Geo &G, int zfast, int i, int j, int k) {
  return zfast ? (size_t)k + (size_t)G.n3 * ((size_t)j + (size_t)G.n2 * i)
               : (size_t)i + (size_t)G.n1 * ((size_t)j + (size_t)G.n2 * k);
}

template <class T>
__device__ __forceinline__ void store_out(const NciOut &O, size_t idx, T crho, T cgrad) {
  if (O.is_f32) {
    ((float *)O.crho)[idx] = (float)crho;
    ((float *)O.cgrad)[idx] = (float)cgrad;
  } else {
    ((double *)O.crho)[idx] = (double)crho;
    ((double *)O.cgrad)[idx] = (double)cgrad;
  }
}

}  // namespace c2
