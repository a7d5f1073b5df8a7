// Truncated SVD split of a small matrix (at most 64 on the shorter side) in
// two launches: Householder QR and one-sided Jacobi in one workgroup's LDS,
// then the left rotations replayed on many.  For pq_decompose's matrices --
// two MPS sites merged over a bond of at most 32 -- the library SVD is some
// 50 to 100 dependent launches (140 to 190 us for 2 x 2, 0.67 ms for 16 x 16,
// 2.4 ms for 64 x 64 complex128, calls included); this takes 30 us, 99 us and
// 0.70 ms.  Errors, as |X - B C| / |X| over random matrices (library in
// brackets): complex128 7.1e-16 (1.4e-15) at 16 x 16 and 1.5e-15 (2.0e-15) at
// 64 x 64, complex64 3.7e-7 (9.1e-7) and 7.3e-7 (1.1e-6); equal at 2 x 2, and
// far smaller on graded spectra (six decades, 16 x 16: 6.9e-16 against
// 8.6e-12).  Singular values and orthogonality likewise.  Only the smallest
// singular values of graded matrices of up to 8 columns are less exact, 0.3 of
// an ulp of the largest against 0.1.
//
//   X (m x n, or its conjugate transpose when m < n) = A (p x q), p >= q
//   A = Q R (Householder);  L = R^H
//   L W = V Sigma with W a product of plane rotations (one-sided Jacobi):
//   A = (Q W) Sigma V^H
//
// QR first: the rotations then act on q x q whatever p is, and a graded
// spectrum -- the rule for MPS bonds -- takes 8 sweeps instead of 20 to 30.
// V Sigma is L itself after the rotations; Q W is Q's rows with the same
// rotations applied, row by row (k_jacobi_left), so the rotations are
// logged and U never passes through the single workgroup.
//
// Jacobi ordering: columns i and i ^ r for every r in 1 .. QP - 1.  Three
// r's that XOR to zero (a line over GF(2)) pair up the same groups of four
// columns, so a group is read into registers once for three rounds: 21 LDS
// passes and barriers per 64-column sweep instead of 63 (the lines are the
// cosets of GF(4)* in GF(64)* and GF(16)*; odd powers of two have no such
// partition and keep a few single r's).  16 lanes hold a group's rows, so
// every inner product is a sum over a DPP row.
// Bound: instruction issue of one wave per SIMD of one CU -- 612 us of the 64
// x 64 call are the one workgroup (8 sweeps of 21 lines, a fifth of it QR),
// 73 the replay.  The round-robin of dependent rounds leaves nothing for
// other CUs.  One rounding per element and rotation (turn, times) costs 6 % of
// that over c x - s y with rounded factors and halves the errors.
#include "pq_jacobi.h"

#include <cmath>
#include <cstring>
#include <utility>

namespace {

// A line as bytes of one word: a, b (the group's columns are c0, c0 ^ a,
// c0 ^ b, c0 ^ a ^ b; their pivot bits: a has ha and not hb, b has hb and
// not ha) and ha + 8 hb + 64 (three rounds a, b, a ^ b; otherwise one, a).
// The kernels keep the lines in LDS: read from their arguments in the loop,
// they would go through the vector memory counter and wait for the log's
// stores.
#define JAC_MAX_LINES 21
#define JAC_LOG 18            // log entries of a group and line: (Re s, Im s, 1 - c) of six rotations
struct Ordering {
  uint32_t line[JAC_MAX_LINES];
  int nline;
};

int top_bit(int v) {
  int h = 0;
  while (v >> (h + 1)) ++h;
  return h;
}

Ordering make_ordering(int qp) {
  static const uint8_t l4[] = {1, 2}, l8[] = {1, 6}, s8[] = {2, 3, 4, 5};
  static const uint8_t l32[] = {1, 2, 4, 8, 5, 10, 6, 16, 7, 18, 9, 17, 11, 20, 13, 19, 14, 23},
                       s32[] = {26, 27, 28, 29};
  Ordering o;
  memset(&o, 0, sizeof(o));
  auto add = [&](int a, int b, int n) {
    if (n == 3) {
      // reduce: distinct top bits, each absent from the other
      if (top_bit(a) == top_bit(b)) b ^= a;
      if (top_bit(a) < top_bit(b)) std::swap(a, b);
      if ((a >> top_bit(b)) & 1) a ^= b;
    } else {
      // any second direction outside a's bits (no single has all of them)
      for (int t = 0; (1 << t) < qp; ++t)
        if (!((a >> t) & 1)) b = 1 << t;
    }
    o.line[o.nline++] = (uint32_t)(a | b << 8 | (top_bit(a) | top_bit(b) << 3 | (n == 3) << 6) << 16);
  };
  auto field = [&](int bits, int poly) {       // lines g^k, g^(k + order / 3)
    const int order = (1 << bits) - 1;
    std::vector<int> pw(order);
    int v = 1;
    for (int k = 0; k < order; ++k) {
      pw[k] = v;
      v <<= 1;
      if (v >> bits) v ^= poly;
    }
    for (int k = 0; k < order / 3; ++k) add(pw[k], pw[k + order / 3], 3);
  };
  if (qp == 4) {
    add(l4[0], l4[1], 3);
  } else if (qp == 8) {
    add(l8[0], l8[1], 3);
    for (int x : s8) add(x, 0, 1);
  } else if (qp == 16) {
    field(4, 0x13);
  } else if (qp == 32) {
    for (int k = 0; k < 18; k += 2) add(l32[k], l32[k + 1], 3);
    for (int x : s32) add(x, 0, 1);
  } else {
    field(6, 0x43);
  }
  return o;
}

// ------------------------------------------------------------ device helpers
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// Sum over the 16 lanes of a DPP row (rotations by 8, 4, 2, 1), in every lane.
template <typename R>
__device__ __forceinline__ R row_sum(R v) {
  v += dpp_mov<0x128>(v);
  v += dpp_mov<0x124>(v);
  v += dpp_mov<0x122>(v);
  v += dpp_mov<0x121>(v);
  return v;
}
__device__ __forceinline__ double rsq_raw(double x) { return __builtin_amdgcn_rsq(x); }
__device__ __forceinline__ float rsq_raw(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rcp_raw(double x) { return __builtin_amdgcn_rcp(x); }
__device__ __forceinline__ float rcp_raw(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double sqrt_raw(double x) { return __builtin_amdgcn_sqrt(x); }
__device__ __forceinline__ float sqrt_raw(float x) { return __builtin_amdgcn_sqrtf(x); }
// 1 / sqrt(x) (x > 0, its square root normal): to a few ulp, and to within
// half an ulp or so by one more step on the exact residual.
__device__ __forceinline__ float rsq_near(float x) { return rsq_raw(x); }
__device__ __forceinline__ double rsq_near(double x) {
  const double y = rsq_raw(x);
  return fma(y, 0.5 * fma(-x * y, y, 1.0), y);
}
template <typename R>
__device__ __forceinline__ R rsq_full(R x) {
  R y = rsq_raw(x);
  y = fma(y, R(0.5) * fma(-x * y, y, R(1)), y);
  const R h = y * y, lo = fma(y, y, -h);
  return fma(y, R(0.5) * (fma(-x, h, R(1)) - x * lo), y);
}
template <typename R>
__device__ __forceinline__ R rcp_full(R x) {
  R y = rcp_raw(x);
  y = fma(y, fma(-x, y, R(1)), y);
  return fma(y, fma(-x, y, R(1)), y);
}

template <typename R> struct Tol;
template <> struct Tol<double> {
  static constexpr double cos2 = 1e-30;    // rotate while |x^H y|^2 > cos2 |x|^2 |y|^2
  static constexpr double done = 1e-17;    // squared angle and cosine that one more sweep would square
  static constexpr double floor2 = 1e-20;  // columns below 1e-10 of the whole are far under any cut-off
  static constexpr double least = 2.3e-308;   // under this a square is subnormal or zero
  static constexpr double zero2 = 1e-250;  // a column's squared norm that counts as zero (largest element 1)
  static constexpr double small2 = 1e-34;  // an element whose square is this part of its column's counts as zero
};
template <> struct Tol<float> {
  static constexpr float cos2 = 9e-14f;
  static constexpr float done = 1e-8f;
  static constexpr float floor2 = 1e-12f;
  static constexpr float least = 1.2e-38f;
  static constexpr float zero2 = 1e-20f;
  static constexpr float small2 = 1e-17f;
};

// Sum over the 8 lanes of a half row, in each of them.
template <typename R>
__device__ __forceinline__ R half_sum(R v) {
  v += dpp_mov<0x141>(v);  // row_half_mirror: l and 7 - l
  v += dpp_mov<0x4e>(v);   // quad_perm 2, 3, 0, 1
  v += dpp_mov<0xb1>(v);   // quad_perm 1, 0, 3, 2
  return v;
}
// x' = c x - s y,  y' = c y + conj(s) x  with c = 1 - k: the change is summed
// first and x added last, so an element is rounded once at its own size
// whatever the number of terms (as c x - s y, three times: the errors of 64
// columns, eight sweeps of 63 rotations each, were 2 times the present ones).
template <typename R, typename C>
__device__ __forceinline__ void turn(C& x, C& y, R sr, R si, R k) {
  const C a = x, b = y;
  x.x = a.x - fma(sr, b.x, fma(-si, b.y, k * a.x));
  x.y = a.y - fma(sr, b.y, fma(si, b.x, k * a.y));
  y.x = b.x + fma(sr, a.x, fma(si, a.y, -k * b.x));
  y.y = b.y + fma(sr, a.y, fma(-si, a.x, -k * b.y));
}

// v (h + l), rounded once: l is what rounding h left of a factor.
__device__ __forceinline__ float times(float v, double h, double) { return (float)((double)v * h); }
__device__ __forceinline__ double times(double v, double h, double l) { return fma(v, h, v * l); }

// The four columns of group g on a line: c0 is the one with both pivot bits
// clear.
__device__ __forceinline__ void group_columns(uint32_t line, int g, int (&col)[4]) {
  const int a = line & 255, b = (line >> 8) & 255, ha = (line >> 16) & 7, hb = (line >> 19) & 7;
  const int lo = ha < hb ? ha : hb, hi = ha < hb ? hb : ha;
  g = ((g >> lo) << (lo + 1)) | (g & ((1 << lo) - 1));
  g = ((g >> hi) << (hi + 1)) | (g & ((1 << hi) - 1));
  col[0] = g;
  col[1] = g ^ a;
  col[2] = g ^ b;
  col[3] = g ^ a ^ b;
}
__device__ __forceinline__ bool three_rounds(uint32_t line) { return (line >> 22) & 1; }

// One round of a group: rotates columns (U, W) and (U2, W2), squared norms
// n, so that each pair's inner product vanishes:
//   x' = c x - s y,  y' = c y + conj(s) x
// A lone wave per SIMD runs a group's rounds one after another, so the time
// is the number of instructions: no branches, and the two pairs share the
// sums and the angle -- lanes 0-7 of the row take the first pair, lanes 8-15
// the second, and swap the results.  A pair that needs no rotation gets s =
// 0, c = 1 (k = 1 - c = 0).
template <typename R, typename C, int LRP, int U, int W, int U2, int W2>
__device__ __forceinline__ void rotate2(C (&x)[4][LRP], R (&n)[4], R fl, bool& big, R* e, int l) {
  R g[2][2];
  constexpr int iu[2] = {U, U2}, iw[2] = {W, W2};
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    R gr = 0, gi = 0;
#pragma unroll
    for (int t = 0; t < LRP; ++t) {
      const C a = x[iu[z]][t], b = x[iw[z]][t];
      gr = t ? fma(a.x, b.x, gr) : a.x * b.x;
      gr = fma(a.y, b.y, gr);
      gi = t ? fma(a.x, b.y, gi) : a.x * b.y;
      gi = fma(-a.y, b.x, gi);
    }
    g[z][0] = gr;
    g[z][1] = gi;
  }
  const bool hi = l >= 8;
  // the first step of the sum leaves each half with its own pair
  R gr = (hi ? g[1][0] : g[0][0]) + dpp_mov<0x128>(hi ? g[0][0] : g[1][0]);
  R gi = (hi ? g[1][1] : g[0][1]) + dpp_mov<0x128>(hi ? g[0][1] : g[1][1]);
  gr = half_sum(gr);
  gi = half_sum(gi);
  const R nu = hi ? n[U2] : n[U], nw = hi ? n[W2] : n[W];
  const R g2 = fma(gr, gr, gi * gi);
  const R nn = fmax(nu, fl) * fmax(nw, fl);
  // (a subnormal g2, which two columns far under the floor can have in
  // float, has no 1 / sqrt: the instruction returns infinity for it)
  const bool rot = g2 > fmax(Tol<R>::cos2 * nn, Tol<R>::least);
  // the angle from raw estimates: any finite s of at most sqrt(1/2) gives a
  // unitary rotation, as k = 1 - c is computed from s itself
  const R ig = rsq_raw(g2);
  const R ze = R(0.5) * (nw - nu) * ig;
  const R ta = rcp_raw(fabs(ze) + sqrt_raw(fma(ze, ze, R(1))));
  const R t = rot ? (ze < 0 ? -ta : ta) : R(0);
  const R ti = rot ? t * ig : R(0);
  const R wr = ti * gr, wi = -ti * gi;
  const R x2 = fma(wr, wr, fma(wi, wi, R(1))), c0 = rsq_near(x2);
  const R sr = c0 * wr, si = c0 * wi, d = ti * g2;
  // k (2 - k) = |s|^2: an estimate, then a Newton step on the residual.  Its
  // error is far below an ulp of 1, so repeated rotations do not scale the
  // columns.
  const R s2 = fma(sr, sr, si * si), k0 = s2 * rcp_raw(R(1) + c0);
  const R k = fma(fma(k0, k0, fma(R(-2), k0, s2)), R(0.5) * x2 * c0, k0);
  big = big || (rot && (g2 > Tol<R>::done * nn || t * t > Tol<R>::done));
  if ((l & 7) == 0) {
    R* q = e + 3 * (l >> 3);
    q[0] = sr;
    q[1] = si;
    q[2] = k;
  }
  const R osr = dpp_mov<0x128>(sr), osi = dpp_mov<0x128>(si), ok = dpp_mov<0x128>(k), od = dpp_mov<0x128>(d);
  const R zr[2] = {hi ? osr : sr, hi ? sr : osr}, zi[2] = {hi ? osi : si, hi ? si : osi},
          zk[2] = {hi ? ok : k, hi ? k : ok}, zd[2] = {hi ? od : d, hi ? d : od};
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    n[iu[z]] = fmax(n[iu[z]] - zd[z], R(0));
    n[iw[z]] += zd[z];
#pragma unroll
    for (int t2 = 0; t2 < LRP; ++t2) turn(x[iu[z]][t2], x[iw[z]][t2], zr[z], zi[z], zk[z]);
  }
}

#define JAC_THREADS 256
#define JAC_GROUPS 16

// One workgroup: X -> A in LDS, QR, L = R^H, the sweeps; writes Q, the
// rotation log, the singular values' order and chi, and the factor that
// holds V.  RP: rows of A per lane (16 lanes per column), QP: columns of L,
// padded with zero columns to a power of two.
template <typename C, int RP, int QP>
__global__ __launch_bounds__(JAC_THREADS) void k_jacobi(JacArgs j, Ordering o) {
  typedef typename real_of<C>::type R;
  constexpr int PP = 16 * RP;                       // padded rows of A
  constexpr int LRP = QP > 16 ? QP / 16 : 1, LR = 16 * LRP;   // padded rows of L
  extern __shared__ __align__(16) unsigned char sm[];
  const int p = j.p, q = j.q;
  C* A = reinterpret_cast<C*>(sm);                  // [q][PP]
  C* L = A + (size_t)q * PP;                        // [QP][LR]
  __shared__ C v0s[JAC_MAX_Q];
  __shared__ double vh[JAC_MAX_Q], vl[JAC_MAX_Q];
  __shared__ R fs[JAC_MAX_Q], nrm[JAC_MAX_Q], red[JAC_THREADS / 64];
  __shared__ int pos[JAC_MAX_Q], busy[2], chi_s;
  __shared__ uint32_t lines[JAC_MAX_LINES];
  const int tid = threadIdx.x, grp = tid / 16, l = tid % 16;

  // ---- X into LDS; its largest magnitude; row / column offsets first (in L)
  {
    int32_t* om = reinterpret_cast<int32_t*>(L);
    int32_t* on = om + j.m;
    for (int i = tid; i < j.m + j.n; i += JAC_THREADS) {
      int32_t a, b;
      if (i < j.m) group_offsets(j.gm, (uint32_t)i, a, b);
      else group_offsets(j.gn, (uint32_t)(i - j.m), a, b);
      om[i] = a;
    }
    __syncthreads();
    const C* X = reinterpret_cast<const C*>(j.X);
    R mx = 0;
    for (int e = tid; e < q * PP; e += JAC_THREADS) {
      const int c = e / PP, r = e % PP;             // A's column and row
      C v;
      v.x = v.y = 0;
      if (r < p) {
        v = j.trans ? X[om[c] + on[r]] : X[om[r] + on[c]];
        if (j.trans) v.y = -v.y;
      }
      A[e] = v;
      mx = fmax(mx, fmax(fabs(v.x), fabs(v.y)));
    }
    for (int w = 32; w > 0; w >>= 1) mx = fmax(mx, __shfl_xor(mx, w));
    if (tid % 64 == 0) red[tid / 64] = mx;
    if (tid == 0) busy[0] = busy[1] = 0;
    if (tid < o.nline) lines[tid] = o.line[tid];
    __syncthreads();
  }
  R mx = red[0];
  for (int w = 1; w < JAC_THREADS / 64; ++w) mx = fmax(mx, red[w]);
  // scale by a power of two, so that squares neither overflow nor vanish
  int ex = 0;
  if (mx > 0) (void)frexp(mx, &ex);
  for (int e = tid; e < q * PP; e += JAC_THREADS) {
    C v = A[e];
    v.x = ldexp(v.x, -ex);
    v.y = ldexp(v.y, -ex);
    A[e] = v;
  }
  for (int e = tid; e < QP * LR; e += JAC_THREADS) L[e].x = L[e].y = 0;
  __syncthreads();

  // ---- QR: H_k = I - f v v^H; v stays below the diagonal, L gets R^H.
  // Column c belongs to lane group c % 16 throughout; a group updates its (at
  // most NC) columns side by side.
  constexpr int NC = QP > 16 ? QP / 16 : 1;
  auto reflect = [&](const C (&v)[RP], R f, int k, bool to_l) {
    C a[NC][RP];
    R wr[NC], wi[NC];
#pragma unroll
    for (int z = 0; z < NC; ++z) {
      const int c = grp + 16 * z;
      wr[z] = wi[z] = 0;
      if (c > k && c < q) {
#pragma unroll
        for (int t = 0; t < RP; ++t) {
          a[z][t] = A[c * PP + l + 16 * t];
          wr[z] = fma(v[t].x, a[z][t].x, fma(v[t].y, a[z][t].y, wr[z]));
          wi[z] = fma(v[t].x, a[z][t].y, fma(-v[t].y, a[z][t].x, wi[z]));
        }
      }
    }
#pragma unroll
    for (int z = 0; z < NC; ++z) {
      wr[z] = f * row_sum(wr[z]);
      wi[z] = f * row_sum(wi[z]);
    }
#pragma unroll
    for (int z = 0; z < NC; ++z) {
      const int c = grp + 16 * z;
      if (c > k && c < q) {
#pragma unroll
        for (int t = 0; t < RP; ++t) {
          // the change first: one rounding at the element's own size
          a[z][t].x -= fma(v[t].x, wr[z], -v[t].y * wi[z]);
          a[z][t].y -= fma(v[t].x, wi[z], v[t].y * wr[z]);
          A[c * PP + l + 16 * t] = a[z][t];
          if (to_l && l + 16 * t == k) {
            L[k * LR + c].x = a[z][t].x;
            L[k * LR + c].y = -a[z][t].y;
          }
        }
      }
    }
  };
  for (int k = 0; k < q; ++k) {
    C v[RP];
    R b2 = 0;                                       // squared norm below the diagonal
#pragma unroll
    for (int t = 0; t < RP; ++t) {
      v[t] = A[k * PP + l + 16 * t];
      if (l + 16 * t <= k) v[t].x = v[t].y = 0;
      b2 = fma(v[t].x, v[t].x, fma(v[t].y, v[t].y, b2));
    }
    const C d = A[k * PP + k];
    b2 = row_sum(b2);
    const R d2 = fma(d.x, d.x, d.y * d.y);
    // H is unitary for any v, as f = 2 / |v|^2 of the very v it is applied
    // with; that H maps the column onto the diagonal decides v.  A column
    // that is zero below the diagonal (under any rounding of the matrix) is
    // left alone; a diagonal element under the rounding of the rest counts
    // as zero, so that its phase is never taken from a square that vanishes.
    const bool some = !(b2 <= Tol<R>::zero2), ang = d2 > Tol<R>::small2 * b2;
    const R n2 = b2 + d2, nx = n2 * rsq_full(n2), id = ang ? rsq_full(d2) : R(0);
    C v0, rd;                                       // rd: the column's element of R
    rd.x = ang ? d.x * id * nx : nx;
    rd.y = ang ? d.y * id * nx : R(0);
    v0.x = !some ? R(0) : (ang ? rd.x + d.x : nx);  // (nx is NaN for a zero column)
    v0.y = some && ang ? rd.y + d.y : R(0);
    const R f = some ? R(2) * rcp_full(fma(v0.x, v0.x, fma(v0.y, v0.y, b2))) : R(0);
    rd.x = some ? -rd.x : d.x;
    rd.y = some ? -rd.y : d.y;
#pragma unroll
    for (int t = 0; t < RP; ++t)
      if (l + 16 * t == k) v[t] = v0;
    reflect(v, f, k, true);
    if (grp == (k & (JAC_GROUPS - 1)) && l == 0) {
      L[k * LR + k].x = rd.x;
      L[k * LR + k].y = -rd.y;
      v0s[k] = v0;
      fs[k] = f;
    }
    __syncthreads();
  }
  // ---- Q = H_0 ... H_{q-1} I in place, last reflector first: every group
  // reads v_k before the barrier, then column k's group overwrites it.
  for (int k = q - 1; k >= 0; --k) {
    const C v0 = v0s[k];
    const R f = fs[k];
    C v[RP];
#pragma unroll
    for (int t = 0; t < RP; ++t) {
      const int r = l + 16 * t;
      v[t] = A[k * PP + r];
      if (r < k) v[t].x = v[t].y = 0;
      if (r == k) v[t] = v0;
    }
    __syncthreads();
    if (grp == (k & (JAC_GROUPS - 1))) {
#pragma unroll
      for (int t = 0; t < RP; ++t) {
        C e;   // e_k - f v conj(v0)
        e.x = (l + 16 * t == k ? R(1) : R(0)) - f * (v[t].x * v0.x + v[t].y * v0.y);
        e.y = -f * (v[t].y * v0.x - v[t].x * v0.y);
        A[k * PP + l + 16 * t] = e;
      }
    }
    reflect(v, f, k, false);
  }
  __syncthreads();
  {
    C* Q = reinterpret_cast<C*>(j.Q);
    for (int e = tid; e < q * p; e += JAC_THREADS) Q[e] = A[(e / p) * PP + e % p];
  }

  // ---- sweeps over L's columns
  constexpr int NG = QP / 4;                        // groups of four columns
  const bool on = grp < NG;
  R* log = reinterpret_cast<R*>(j.log);
  int sweep = 0;
  bool more = true;
  for (; more && sweep < JAC_MAX_SWEEPS; ++sweep) {
    R fl = 0;
    for (int c = grp; c < QP; c += JAC_GROUPS) {    // the columns' squared norms
      R n2 = 0;
#pragma unroll
      for (int t = 0; t < LRP; ++t) {
        const C a = L[c * LR + l + 16 * t];
        n2 += a.x * a.x + a.y * a.y;
      }
      n2 = row_sum(n2);
      if (l == 0) nrm[c] = n2;
    }
    __syncthreads();
    for (int c = 0; c < QP; ++c) fl += nrm[c];
    fl *= Tol<R>::floor2;
    // every lane has read the last sweep's flag by the barrier above
    if (tid == 0) busy[(sweep + 1) & 1] = 0;
    __syncthreads();
    bool big = false;
    for (int s = 0; s < o.nline; ++s) {
      if (on) {
        const uint32_t ln = __builtin_amdgcn_readfirstlane(lines[s]);
        int col[4];
        group_columns(ln, grp, col);
        C x[4][LRP];
        R n[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          n[u] = nrm[col[u]];
#pragma unroll
          for (int t = 0; t < LRP; ++t) x[u][t] = L[col[u] * LR + l + 16 * t];
        }
        R* e = log + (((size_t)sweep * o.nline + s) * NG + grp) * JAC_LOG;
        // columns (0, 1) and (2, 3), then (0, 2) and (1, 3), (0, 3) and (1, 2)
        rotate2<R, C, LRP, 0, 1, 2, 3>(x, n, fl, big, e, l);
        if (three_rounds(ln)) {
          rotate2<R, C, LRP, 0, 2, 1, 3>(x, n, fl, big, e + 6, l);
          rotate2<R, C, LRP, 0, 3, 1, 2>(x, n, fl, big, e + 12, l);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          if (l == 0) nrm[col[u]] = n[u];
#pragma unroll
          for (int t = 0; t < LRP; ++t) L[col[u] * LR + l + 16 * t] = x[u][t];
        }
      }
      __syncthreads();
    }
    if (big) busy[sweep & 1] = 1;
    __syncthreads();
    more = busy[sweep & 1] != 0;
  }

  // ---- singular values, their order, the bond dimension
  for (int c = grp; c < QP; c += JAC_GROUPS) {
    R n2 = 0;
#pragma unroll
    for (int t = 0; t < LRP; ++t) {
      const C a = L[c * LR + l + 16 * t];
      n2 += a.x * a.x + a.y * a.y;
    }
    n2 = row_sum(n2);
    if (l == 0) nrm[c] = sqrt(n2);
  }
  __syncthreads();
  if (tid < q) {
    const R mine = nrm[tid];
    int at = 0;
    for (int c = 0; c < q; ++c) at += nrm[c] > mine || (nrm[c] == mine && c < tid);
    pos[tid] = at;
  }
  if (tid == 0) {
    double norm = 0.0;
    for (int c = 0; c < q; ++c) norm += (double)nrm[c] * (double)nrm[c];
    norm = sqrt(norm);
    int chi = 0;
    for (int c = 0; c < q; ++c)
      if ((double)nrm[c] / norm > j.thr) ++chi;
    if (j.max_rank > 0 && chi > j.max_rank) chi = j.max_rank;
    chi_s = chi;
    // the sweeps did not converge (or met infinities or NaN)
    j.host[1] = more || !(norm < INFINITY) ? 1 : 0;
    j.host[0] = chi;
    __threadfence_system();
  }
  __syncthreads();
  const int chi = chi_s;
  JacMeta* meta = reinterpret_cast<JacMeta*>(j.meta);
  if (tid < q) {
    const double sg = (double)nrm[tid], x = ldexp(sg, ex), rt = sqrt(x), rl = fma(-rt, rt, x) / (2 * rt);
    meta->pos[tid] = pos[tid];
    meta->root[tid] = rt;
    meta->rest[tid] = rl;
    vh[tid] = rt / sg;                              // V sqrt(sigma) = L x (vh + vl)
    vl[tid] = (fma(-vh[tid], sg, rt) + rl) / sg;
  }
  if (tid == 0) {
    meta->chi = chi;
    meta->lines = sweep * o.nline;
  }
  __syncthreads();
  // ---- the factor with V = L / sigma: sqrt(sigma) V^H (rows) or V sqrt(sigma)
  C* out = reinterpret_cast<C*>(j.trans ? j.B : j.C);
  for (int e = tid; e < q * q; e += JAC_THREADS) {
    const int c = e / q, r = e % q, at = pos[c];
    if (at >= chi) continue;
    C v = L[c * LR + r];
    v.x = times(v.x, vh[c], vl[c]);
    v.y = times(j.trans ? v.y : -v.y, vh[c], vl[c]);
    out[j.trans ? r + (int64_t)j.m * at : at + (int64_t)chi * r] = v;
  }
}

// U = Q W: Q's rows with the logged rotations applied.  A lane holds one
// group's four columns of a row, so a line's three rounds need no exchange
// (a column per lane and a shuffle per round: 79 us at 64 columns); between
// lines the row passes through LDS.  One wave per workgroup, QP / 4 lanes a
// row; the next line's rotations are loaded while one line is applied.
template <typename C, int QP>
__global__ __launch_bounds__(64) void k_jacobi_left(JacArgs j, Ordering o) {
  typedef typename real_of<C>::type R;
  constexpr int NG = QP / 4, ROWS = 64 / NG;
  __shared__ C buf[ROWS][QP + 1];
  __shared__ uint32_t line[JAC_MAX_LINES];
  const int lane = threadIdx.x, grp = lane % NG, lr = lane / NG, row = blockIdx.x * ROWS + lr;
  const JacMeta* meta = reinterpret_cast<const JacMeta*>(j.meta);
  const int lines = meta->lines, chi = meta->chi;
  if (lane < o.nline) line[lane] = o.line[lane];
  for (int c = grp; c < QP; c += NG) {
    C v;
    v.x = v.y = 0;
    if (row < j.p && c < j.q) v = reinterpret_cast<const C*>(j.Q)[row + (int64_t)j.p * c];
    buf[lr][c] = v;
  }
  __syncthreads();
  const R* log = reinterpret_cast<const R*>(j.log) + (size_t)grp * JAC_LOG;
  constexpr int PF = 4;                             // lines in flight
  R nx[PF][JAC_LOG];
  auto load = [&](int s, R (&e)[JAC_LOG]) {
    s = s < lines ? s : lines - 1;
#pragma unroll
    for (int u = 0; u < JAC_LOG; ++u) e[u] = log[(size_t)s * NG * JAC_LOG + u];
  };
#pragma unroll
  for (int u = 0; u < PF; ++u) load(u, nx[u]);
  for (int s0 = 0, k = 0; s0 < lines; s0 += PF) {
#pragma unroll
    for (int v = 0; v < PF; ++v) {
      if (s0 + v >= lines) break;
      const uint32_t ln = __builtin_amdgcn_readfirstlane(line[k]);
      k = k + 1 == o.nline ? 0 : k + 1;
      int col[4];
      group_columns(ln, grp, col);
      C x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = buf[lr][col[u]];
      const R* e = nx[v];
      turn(x[0], x[1], e[0], e[1], e[2]);
      turn(x[2], x[3], e[3], e[4], e[5]);
      if (three_rounds(ln)) {
        turn(x[0], x[2], e[6], e[7], e[8]);
        turn(x[1], x[3], e[9], e[10], e[11]);
        turn(x[0], x[3], e[12], e[13], e[14]);
        turn(x[1], x[2], e[15], e[16], e[17]);
      }
      load(s0 + v + PF, nx[v]);
#pragma unroll
      for (int u = 0; u < 4; ++u) buf[lr][col[u]] = x[u];
      __syncthreads();
    }
  }
  if (row >= j.p) return;
  C* out = reinterpret_cast<C*>(j.trans ? j.C : j.B);
  for (int c = grp; c < j.q; c += NG) {
    const int at = meta->pos[c];
    if (at >= chi) continue;
    C v = buf[lr][c];
    const double h = meta->root[c], l = meta->rest[c];
    v.x = times(v.x, h, l);
    v.y = times(j.trans ? -v.y : v.y, h, l);
    out[j.trans ? at + (int64_t)chi * row : row + (int64_t)j.m * at] = v;
  }
}

int pad_q(int q) { return q <= 4 ? 4 : (q <= 8 ? 8 : (q <= 16 ? 16 : (q <= 32 ? 32 : 64))); }
int pad_rp(int p) { return p <= 16 ? 1 : (p <= 64 ? 4 : (p <= 128 ? 8 : 16)); }

template <typename C, int RP, int QP>
hipError_t launch_both(const JacArgs& j, const Ordering& o, size_t lds, hipStream_t s) {
  hipLaunchKernelGGL((k_jacobi<C, RP, QP>), dim3(1), dim3(JAC_THREADS), lds, s, j, o);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  constexpr int rows = 64 / (QP / 4);
  hipLaunchKernelGGL((k_jacobi_left<C, QP>), dim3((unsigned)((j.p + rows - 1) / rows)), dim3(64), 0, s, j, o);
  return hipGetLastError();
}

template <typename C, int RP>
hipError_t launch_q(const JacArgs& j, const Ordering& o, size_t lds, hipStream_t s) {
  switch (pad_q(j.q)) {
    case 4: return launch_both<C, RP, 4>(j, o, lds, s);
    case 8: return launch_both<C, RP, 8>(j, o, lds, s);
    case 16: return launch_both<C, RP, 16>(j, o, lds, s);
    case 32: return launch_both<C, RP, 32>(j, o, lds, s);
    default: return launch_both<C, RP, 64>(j, o, lds, s);
  }
}

size_t lds_bytes(int p, int q, size_t es) {
  const int qp = pad_q(q);
  return ((size_t)q * 16 * pad_rp(p) + (size_t)qp * std::max(qp, 16)) * es;
}

}  // namespace

// LDS of one workgroup, less the static arrays of k_jacobi
#define JAC_LDS_BYTES (152 * 1024)

bool jacobi_fits(int64_t m, int64_t n, size_t es) {
  const int64_t p = std::max(m, n), q = std::min(m, n);
  if (q < 1 || q > JAC_MAX_Q || p > 256) return false;
  // the offsets of X's rows and columns pass through L, which is small for few
  // columns
  const int qp = pad_q((int)q);
  if ((size_t)(m + n) * 4 > (size_t)qp * std::max(qp, 16) * es) return false;
  return lds_bytes((int)p, (int)q, es) <= JAC_LDS_BYTES;
}

size_t jacobi_log_bytes(int64_t q, size_t es) {
  const int qp = pad_q((int)q);
  return (size_t)JAC_MAX_SWEEPS * JAC_MAX_LINES * (qp / 4) * JAC_LOG * (es / 2);
}

template <typename C>
hipError_t launch_jacobi(JacArgs j, hipStream_t s) {
  static const Ordering o4 = make_ordering(4), o8 = make_ordering(8), o16 = make_ordering(16), o32 = make_ordering(32),
                        o64 = make_ordering(64);
  j.trans = j.m < j.n ? 1 : 0;
  j.p = std::max(j.m, j.n);
  j.q = std::min(j.m, j.n);
  const int qp = pad_q(j.q);
  const Ordering& o = qp == 4 ? o4 : (qp == 8 ? o8 : (qp == 16 ? o16 : (qp == 32 ? o32 : o64)));
  const size_t lds = lds_bytes(j.p, j.q, sizeof(C));
  switch (pad_rp(j.p)) {
    case 1: return launch_q<C, 1>(j, o, lds, s);
    case 4: return launch_q<C, 4>(j, o, lds, s);
    case 8: return launch_q<C, 8>(j, o, lds, s);
    default: return launch_q<C, 16>(j, o, lds, s);
  }
}
template hipError_t launch_jacobi<c128>(JacArgs, hipStream_t);
template hipError_t launch_jacobi<c64>(JacArgs, hipStream_t);
