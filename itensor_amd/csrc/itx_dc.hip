// Divide and conquer for the symmetric tridiagonal eigenproblem, batched over
// matrices, entirely on the device.
//
// Method: Cuppen (Numer. Math. 36 (1981) 177) tears T into two halves plus a
// rank-one term; the merged problem D + rho z z^T has as eigenvalues the
// roots of the secular equation 1 + rho sum z_i^2 / (d_i - x) = 0 (Golub,
// SIAM Rev. 15 (1973) 318), found by rational interpolation of the two
// halves of the sum (Bunch, Nielsen & Sorensen, Numer. Math. 31 (1978) 31)
// inside a bracket; the eigenvectors come from the z for which the computed
// roots are exact (Gu & Eisenstat, SIAM J. Matrix Anal. Appl. 15 (1994)
// 1266), so they are orthogonal to working precision without further care.
// Entries of z that are negligible and pairs of nearly equal d are deflated
// first (Dongarra & Sorensen, SIAM J. Sci. Stat. Comput. 8 (1987) s139).
//
// The tearing goes down to single rows: the n rows are cut into L = 2^p >= n
// leaves of one or no row, node t of level l covers the rows
// [t 2^l n / L, (t+1) 2^l n / L), rounded down.  Nodes up to 64 rows are merged by
// one workgroup with everything in LDS; above, every level is four launches
// over the merges of all matrices: preparation (sort, deflation), roots,
// vectors of the secular problem, and the product of the children's
// vectors with them on the FP64 matrix cores.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "itx_tri.h"

namespace itx {
namespace {

constexpr double DC_EPS = DBL_EPSILON / 2;
constexpr int SB = 64;         // rows of an LDS-resident subtree
constexpr int SBP = SB + 1;    // LDS column pitch
constexpr int ST = 256;        // its threads: four per row

// first row of node t of level l of a matrix of order n with 2^p leaves
__device__ __forceinline__ int node_row(int t, int l, int n, int p) {
  return int((unsigned(t * n) << l) >> p);  // at most 2^18
}
// the node of level l that holds row e
__device__ __forceinline__ int node_of(int e, int l, int n, int p) {
  return int(((unsigned(e + 1) << p) - 1u) / (unsigned(n) << l));
}

// ---- one root of the secular equation ----------------------------------------
// Poles d[0..k) ascending, weights w_i = rho z_i^2 > 0 (weight(i));
// root j lies between d[j] and d[j+1] (the last one between d[k-1] and
// d[k-1] + sum w).  sums(d_K, mu) returns over all poles, with del_i =
// (d_i - d_K) - mu, the sums of w/del and w/del^2 separately for negative
// and positive del: the poles below and above the root.  The root is d[K] +
// mu with K the nearer pole, so every del_i is accurate.
struct SecSums {
  double p, pp, f, fp;  // psi, psi' (below), phi, phi' (above)
};
// A step interpolates the sums below and above by one pole each, at d[j] and
// d[j+1]; after the first one the nearer pole keeps its own weight (the
// fixed-weight method: Li, LAPACK Working Note 89 (1993)), which converges in
// one step less: 4 evaluations on average.  A step below 1e-8 of mu is the last one: the next would be of
// the order of its square.
template <class Weight, class Sums>
__device__ __forceinline__ void secular_root(int j, int k, const double *d, double wsum, Weight weight, Sums sums,
                                             int &K, double &mu) {
  const bool last = j == k - 1;
  K = j;
  if (k == 1) {
    mu = wsum;
    return;
  }
  const int split = last ? k - 2 : j;
  const double gap = last ? wsum : d[j + 1] - d[j];
  double lo = 0.0, hi = gap;
  mu = 0.5 * gap;
  double dK = d[j];
  SecSums s = sums(dK, mu);
  double f = 1.0 + (s.p + s.f);
  if (!last && f < 0.0) {  // nearer to the upper pole
    K = j + 1;
    dK = d[K];
    mu -= gap;
    lo = mu;
    hi = 0.0;
  }
  const double d1 = d[split] - dK, d2 = d[split + 1] - dK, wK = weight(last ? k - 1 : K);
  for (int it = 0; it < 100; ++it) {
    // the error of the sums is a few eps of the sum of the terms' sizes, and
    // the last bit of mu moves them by eps mu times their derivative
    if (fabs(f) <= DC_EPS * (8.0 * (1.0 + fabs(s.p) + fabs(s.f)) + fabs(mu) * (s.pp + s.fp))) break;
    if (f < 0.0)
      lo = fmax(lo, mu);
    else
      hi = fmin(hi, mu);
    if (hi - lo <= 2.0 * DC_EPS * fmax(fabs(lo), fabs(hi))) break;
    const double e1 = d1 - mu, e2 = d2 - mu;
    if (last) {  // its neighbour above is the last pole, whose term psi holds too
      const double r = fast_rcp(e2);
      s.fp = wK * r * r;
      s.pp = fmax(s.pp - s.fp, 0.0);
    }
    double c = f - e1 * s.pp - e2 * s.fp;
    if (!last && it > 0) {
      const bool low = K == j;
      const double near = fast_rcp(low ? e1 : e2), g = gap * wK * near * near;
      c = f - (low ? e2 : e1) * (s.pp + s.fp) + (low ? g : -g);
    }
    const double a = (e1 + e2) * f - e1 * e2 * (s.pp + s.fp), b = e1 * e2 * f;
    // the root of c eta^2 - a eta + b between the two poles (last: above both)
    const double sg = last ? -1.0 : 1.0, q = sg * fast_sqrt(a * a - 4.0 * b * c), r = a - q, t = a + q;
    const bool first = sg * a <= 0.0;
    double x = mu + (first ? r : 2.0 * b) * fast_rcp(first ? 2.0 * c : t);
    const bool inside = x > lo && x < hi;
    if (!inside) x = 0.5 * (lo + hi);
    if (x == mu || x == 0.0) break;
    const bool small = inside && fabs(x - mu) <= 1e-8 * fabs(x);
    mu = x;
    if (small) break;
    s = sums(dK, mu);
    f = 1.0 + (s.p + s.f);
  }
}
// one pole's terms: negative ones to psi, positive ones to phi
__device__ __forceinline__ void secular_term(double del, double w, SecSums &s) {
  const double r = fast_rcp(del), t = w * r, lo = fmin(t, 0.0), up = fmax(t, 0.0);
  s.p += lo;
  s.f += up;
  s.pp = fma(lo, r, s.pp);
  s.fp = fma(up, r, s.fp);
}

// ---- deflation -----------------------------------------------------------------
// Entries with rho |z| <= tol leave the secular problem as they are (tol: 8
// eps of the largest |d|, or of a quarter: z has norm 1); of two neighbours in the order of d whose
// difference is as negligible, a rotation of their columns zeroes one z.
__device__ __forceinline__ bool near_pair(double d0, double z0, double d1, double z1, double tol) {
  return fabs((d1 - d0) * z0 * z1) <= tol * (z0 * z0 + z1 * z1);
}
// One thread walks the kept entries (d, z, column), m of them, where some
// pair is near: those that stay in the secular problem go to the front of
// (od, oz, oc), the others to its end; the rotations are recorded in order.
template <class Rot>
__device__ __forceinline__ int deflate(int m, double tol, const double *d, const double *z, const int *col, double *od,
                                       double *oz, int *oc, Rot rot, int &nrot) {
  int k = 0, nd = 0;
  nrot = 0;
  double dp = d[0], zp = z[0];
  int cp = col[0];
  double dn = m > 1 ? d[1] : 0.0, zn = m > 1 ? z[1] : 0.0;
  int cn = m > 1 ? col[1] : 0;
  for (int i = 1; i < m; ++i) {
    const double dj = dn, zj = zn;
    const int cj = cn;
    if (i + 1 < m) {
      dn = d[i + 1];
      zn = z[i + 1];
      cn = col[i + 1];
    }
    if (near_pair(dp, zp, dj, zj, tol)) {
      const double r = sqrt(zj * zj + zp * zp), c = zj / r, s = -zp / r;
      rot(nrot++, cp, cj, c, s);
      ++nd;
      od[m - nd] = dp * c * c + dj * s * s;
      oc[m - nd] = cp;
      dp = dp * s * s + dj * c * c;
      zp = r;
    } else {
      od[k] = dp;
      oz[k] = zp;
      oc[k] = cp;
      ++k;
      dp = dj;
      zp = zj;
    }
    cp = cj;
  }
  od[k] = dp;
  oz[k] = zp;
  oc[k] = cp;
  return k + 1;
}

__device__ __forceinline__ double quad_sum(double v) {
  v += dpp_move<DPP_XOR1>(v);
  return v + dpp_move<DPP_XOR2>(v);
}
__device__ __forceinline__ int quad_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, DPP_XOR1, 0xF, 0xF, true);
  return v + __builtin_amdgcn_update_dpp(0, v, DPP_XOR2, 0xF, 0xF, true);
}
__device__ __forceinline__ double quad_product(double v) {
  v *= dpp_move<DPP_XOR1>(v);
  return v * dpp_move<DPP_XOR2>(v);
}

// root j of a merge in LDS, four threads per root with NT poles each
template <int NT>
__device__ __forceinline__ void small_root(int j, int k, int part, const double *dd, const double *ww, double *dl,
                                           double *lam) {
  double d[NT], w[NT], wt = 0.0;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int a = part + 4 * t;
    d[t] = a < k ? dd[a] : 4.0;  // no pole: away from every root, weight 0
    w[t] = a < k ? ww[a] : 0.0;
    wt += w[t];
  }
  wt = quad_sum(wt);
  int K;
  double mu;
  auto sums = [&](double dK, double mu2) {
    SecSums s{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < NT; ++t) secular_term((d[t] - dK) - mu2, w[t], s);
    s.p = quad_sum(s.p);
    s.pp = quad_sum(s.pp);
    s.f = quad_sum(s.f);
    s.fp = quad_sum(s.fp);
    return s;
  };
  secular_root(j, k, dd, wt, [&](int a) { return ww[a]; }, sums, K, mu);
  const double dK = dd[K];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int a = part + 4 * t;
    if (a < k) dl[a] = (d[t] - dK) - mu;
  }
  if (part == 0) *lam = dK + mu;
}

// ---- subtrees of at most 64 rows -------------------------------------------------
// Per level: every row has four threads.  Bound by the latency of the level's
// dependent phases (the walk over a merge of 64, some six evaluations of the
// secular equation), not by arithmetic: the product of 64 x 64 vectors takes
// 64 MFMAs a wave.
__device__ __forceinline__ void dc_small_run(const DcTask &tk, int sub, double *__restrict__ W,
                                             int *__restrict__ status) {
  __shared__ double Qa[SB * SBP], Qb[SB * SBP], DL[SB * SBP];
  __shared__ double D[SB], Z[SB], ds[SB], zs[SB], dk[SB], zk[SB], Dn[SB], ws[SB], zh[SB];
  __shared__ double rc[SB], rs[SB];
  __shared__ int pm[SB], sel[SB], rp[SB], rq[SB], kof[SB], nrt[SB], wspan[2 * (SB / 16)];
  __shared__ int2 seg[SB];
  const int n = tk.n, p = tk.p;  // subtree `sub` of level min(p, 6)
  const int top = min(p, 6);
  const int r0 = node_row(sub, top, n, p), cnt = node_row(sub + 1, top, n, p) - r0;
  const int tid = threadIdx.x, i = tid >> 2, part = tid & 3, lane = tid & 63, wave = tid >> 6;
  const double *dv = W + tk.d_off, *ev = dv + n;
  double *aux = W + tk.x_off;

  // the scale of T: its largest entry as a power of two, the same for every subtree
  double mx = 0.0;
  bool nan = false;
  for (int e = lane; e < n; e += 64) {
    const double a = fabs(dv[e]), b = fabs(ev[e]);
    nan = nan || a != a || b != b;
    mx = fmax(mx, fmax(a, b));
  }
  // not a number: no decomposition, except that a single row is its own
  nan = __any(nan) && n > 1;
  if (nan && tid == 0) atomicMax(status, 1);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
  // beside an infinite entry every coupling is negligible: d as it stands
  const bool loose = nan || !(mx <= DBL_MAX) || n == 1;
  int ex = 0;
  if (mx > 0.0 && !loose) (void)frexp(mx, &ex);
  ex = min(ex, 1023);  // 2^ex is a number too
  auto diagonal = [&](int g) { return loose ? (nan ? 0.0 : dv[g]) : ldexp(dv[g], -ex); };
  auto coupling = [&](int g) { return loose ? 0.0 : ldexp(ev[g], -ex); };
  if (sub == 0 && tid == 0) aux[AUX_SCALE(n)] = loose ? INFINITY : ldexp(1.0, ex);

  for (int x = tid; x < SB * SBP; x += ST) {
    Qa[x] = (x / SBP == x % SBP) ? 1.0 : 0.0;
    Qb[x] = 0.0;
  }
  if (part == 0) {
    double v = 0.0;
    if (i < cnt) {  // every boundary is torn: the diagonal loses both neighbours' |e|
      const int g = r0 + i;
      v = diagonal(g) - (g > 0 ? fabs(coupling(g - 1)) : 0.0) - (g + 1 < n ? fabs(coupling(g)) : 0.0);
    }
    D[i] = v;
  }
  __syncthreads();

  double *Qo = Qa, *Qn = Qb;
  for (int l = 1; l <= top; ++l) {
    const bool in = i < cnt;
    int ms = 0, me = 0, md = 0;
    double beta = 0.0;
    if (in) {
      const int t = node_of(r0 + i, l, n, p);
      ms = node_row(t, l, n, p) - r0;
      me = node_row(t + 1, l, n, p) - r0;
      md = node_row(2 * t + 1, l - 1, n, p) - r0;
      if (md > ms && md < me) beta = coupling(r0 + md - 1);
    }
    // the rows of the merges that a wave's 16 columns belong to
    if (part == 0 && (i & 15) == 0) wspan[2 * (i >> 4)] = in ? ms : SB;
    if (part == 0 && in && ((i & 15) == 15 || i == cnt - 1)) wspan[2 * (i >> 4) + 1] = me;
    if (part == 0 && !in && (i & 15) == 0) wspan[2 * (i >> 4) + 1] = 0;
    const int m = me - ms;
    const double rho = 2.0 * fabs(beta);
    // z: last row of the upper vectors, first row of the lower ones
    double zi = 0.0;
    if (in && beta != 0.0) {
      zi = i < md ? Qo[i * SBP + md - 1] : Qo[i * SBP + md];
      if (i >= md && beta < 0.0) zi = -zi;
      zi *= 0.70710678118654752440;
    }
    const double di = in ? D[i] : 0.0;
    int rk = 0;
    if (in)
#pragma unroll 4
      for (int j = ms + part; j < me; j += 4) {
        const double dj = D[j];
        rk += (dj < di) || (dj == di && j < i);
      }
    rk = quad_sum(rk);
    if (in && part == 0) {
      ds[ms + rk] = di;
      zs[ms + rk] = zi;
      pm[ms + rk] = i;
      seg[i] = make_int2(ms, me);
      zk[i] = rho;
    }
    __syncthreads();
    if (wave != 0) {
      for (int x = tid - 64; x < SB * SBP; x += ST - 64) DL[x] = 0.0;
    } else if (lane < cnt) {
      // sorted entry `lane`: does its z keep it (z has norm 1), and how many
      // of its merge before it are kept
      const int s0 = seg[lane].x, s1 = seg[lane].y;
      const double dl = ds[lane], zl = zs[lane], rl = zk[lane];  // rl: the merge's rho
      const double tol = 8.0 * DC_EPS * fmax(0.25, fmax(fabs(ds[s0]), fabs(ds[s1 - 1])));
      const int col = pm[lane];
      const bool keep = rl * fabs(zl) > tol;
      const unsigned long long all = __ballot(keep);
      const unsigned long long mine = (all >> s0) & (s1 - s0 == 64 ? ~0ull : (1ull << (s1 - s0)) - 1);
      const int before = __popcll(mine & ((1ull << (lane - s0)) - 1)), kept = __popcll(mine);
      const int at = keep ? s0 + before : s1 - 1 - (lane - s0 - before);
      __builtin_amdgcn_wave_barrier();  // every rho is read before z takes its place
      dk[at] = dl;
      zk[at] = zl;
      sel[at] = col;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const int c = lane - s0;
      const bool near = c + 1 < kept && near_pair(dk[lane], zk[lane], dk[lane + 1], zk[lane + 1], tol);
      const unsigned long long nears = __ballot(near) >> s0;
      if (c == 0) {
        int k = kept, nr = 0;
        if (nears & (s1 - s0 == 64 ? ~0ull : (1ull << (s1 - s0)) - 1)) {
          for (int x = 0; x < kept; ++x) {  // the walk needs its input apart from its output
            ds[s0 + x] = dk[s0 + x];
            zs[s0 + x] = zk[s0 + x];
            pm[s0 + x] = sel[s0 + x];
          }
          k = deflate(kept, tol, ds + s0, zs + s0, pm + s0, dk + s0, zk + s0, sel + s0,
                      [&](int t, int a, int b, double cs, double sn) {
                        rp[s0 + t] = a;
                        rq[s0 + t] = b;
                        rc[s0 + t] = cs;
                        rs[s0 + t] = sn;
                      },
                      nr);
        }
        kof[s0] = k;
        nrt[s0] = nr;
      }
    }
    __syncthreads();
    const int k = in ? kof[ms] : 0, j = i - ms;
    // the rotations, one row of the vectors per thread
    if (in && part == 0) {
      const int nr = nrt[ms];
      for (int t = 0; t < nr; ++t) {
        double *qp = Qo + rp[ms + t] * SBP + i, *qq = Qo + rq[ms + t] * SBP + i;
        const double c = rc[ms + t], s = rs[ms + t], a = *qp, b = *qq;
        *qp = c * a + s * b;
        *qq = c * b - s * a;
      }
    }
    if (in && part == 0 && j < k) ws[i] = rho * zk[i] * zk[i];
    __syncthreads();
    // roots: four threads each
    const bool sec = in && j < k;
    if (sec) {
      const double *dd = dk + ms, *ww = ws + ms;
      if (l <= 4)
        small_root<4>(j, k, part, dd, ww, DL + i * SBP + ms, Dn + i);
      else
        small_root<16>(j, k, part, dd, ww, DL + i * SBP + ms, Dn + i);
    } else if (in && part == 0) {
      Dn[i] = dk[i];
      DL[i * SBP + i] = 1.0;
    }
    __syncthreads();
    // the z for which these roots are exact
    {
      double pr = 1.0;
      if (sec)
#pragma unroll 4
        for (int a = part; a < k; a += 4) {
          const double del = DL[(ms + a) * SBP + i];
          pr *= a == j ? -del : del * fast_rcp(dk[i] - dk[ms + a]);
        }
      pr = quad_product(pr);
      if (sec && part == 0) zh[i] = copysign(sqrt(fmax(pr, 0.0)), zk[i]);
    }
    __syncthreads();
    // column j of the secular problem's vectors
    {
      double nn = 0.0;
      if (sec)
#pragma unroll 4
        for (int a = part; a < k; a += 4) {
          const double v = zh[ms + a] * fast_rcp(DL[i * SBP + ms + a]);
          DL[i * SBP + ms + a] = v;
          nn += v * v;
        }
      nn = quad_sum(nn);
      if (sec) {
        const double f = fast_rsqrt(nn);
#pragma unroll 4
        for (int a = part; a < k; a += 4) DL[i * SBP + ms + a] *= f;
      }
    }
    __syncthreads();
    // Qn(:, c) = sum_l Qo(:, sel(l)) DL(l, c): wave w the columns 16 w ..,
    // rows and l over the merges of these columns (zero elsewhere)
    {
      typedef double v4 __attribute__((ext_vector_type(4)));
      const int cc = 16 * wave + (lane & 15);
      const int llo = wspan[2 * wave], lhi = wspan[2 * wave + 1];
      const int b0 = llo & ~15, nb = max(0, (lhi - b0 + 15) >> 4);  // 16-wide blocks
      auto product = [&](auto blocks) __attribute__((always_inline)) {
        constexpr int NB = decltype(blocks)::value;
        v4 acc[NB];
#pragma unroll
        for (int a = 0; a < NB; ++a) acc[a] = v4{0, 0, 0, 0};
        for (int lb = 0; lb < NB; ++lb) {
          double bq[4], aq[4][NB];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int li = b0 + 16 * lb + 4 * q + (lane >> 4);
            const int sl = li < cnt ? sel[li] : li;
            bq[q] = DL[cc * SBP + li];
#pragma unroll
            for (int a = 0; a < NB; ++a) aq[q][a] = Qo[sl * SBP + b0 + 16 * a + (lane & 15)];
          }
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int a = 0; a < NB; ++a)  // MFMA rows: columns c, MFMA columns: rows of Q
              acc[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(bq[q], aq[q][a], acc[a], 0, 0, 0);
        }
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            Qn[(16 * wave + (lane >> 4) + 4 * r) * SBP + b0 + 16 * a + (lane & 15)] = acc[a][r];
      };
      if (nb == 1)
        product(std::integral_constant<int, 1>{});
      else if (nb == 2)
        product(std::integral_constant<int, 2>{});
      else if (nb == 3)
        product(std::integral_constant<int, 3>{});
      else if (nb == 4)
        product(std::integral_constant<int, 4>{});
    }
    if (part == 0 && in) D[i] = Dn[i];
    double *t = Qo;
    Qo = Qn;
    Qn = t;
    __syncthreads();
  }
  double *Q = W + tk.q_off;
  for (int x = tid; x < SB * SB; x += ST) {
    const int c = x / SB, r = x % SB;
    if (c < cnt && r < cnt) Q[size_t(r0 + c) * n + r0 + r] = Qo[c * SBP + r];
  }
  if (part == 0 && i < cnt) aux[AUX_D(n, 0) + r0 + i] = D[i];
}

__global__ __launch_bounds__(ST) void k_dc_small(const DcTask *__restrict__ tasks, const int2 *__restrict__ blocks,
                                                 double *__restrict__ W, int *__restrict__ status) {
  const int2 bk = blocks[blockIdx.x];
  const DcTask tk = tasks[bk.x];
  dc_small_run(tk, bk.y, W, status + bk.x);
}

// ---- merges above 64 rows ---------------------------------------------------------
constexpr int PT = 512;

// sort, deflation, rotations: one workgroup per merge (level l, node bk.y)
__global__ __launch_bounds__(PT) void k_dc_prep(const DcTask *__restrict__ tasks, const int2 *__restrict__ blocks,
                                                double *__restrict__ W, int l) {
  __shared__ double D[DC_MAX], Z[DC_MAX], ds[DC_MAX], zs[DC_MAX], rc[DC_MAX], rs[DC_MAX];
  __shared__ double wred[PT / 64];
  __shared__ int pm[DC_MAX], pk[DC_MAX], rp[DC_MAX], rq[DC_MAX], wcnt[PT / 64], sh[2];
  const int2 bk = blocks[blockIdx.x];
  const DcTask tk = tasks[bk.x];
  const int n = tk.n, p = tk.p, par = (l - 7) & 1, tid = threadIdx.x;
  const int r0 = node_row(bk.y, l, n, p), m = node_row(bk.y + 1, l, n, p) - r0;
  const int md = node_row(2 * bk.y + 1, l - 1, n, p) - r0;
  double *aux = W + tk.x_off;
  double *Q = W + tk.q_off + (par ? size_t(n) * n : 0) + size_t(r0) * n + r0;  // the merge's block
  const double *Dg = aux + AUX_D(n, par) + r0;
  const double scale = aux[AUX_SCALE(n)];
  const double beta = scale <= DBL_MAX ? W[tk.d_off + n + r0 + md - 1] / scale : 0.0, rho = 2.0 * fabs(beta);
  for (int i = tid; i < m; i += PT) {
    double z = Q[size_t(i) * n + (i < md ? md - 1 : md)] * 0.70710678118654752440;
    if (i >= md && beta < 0.0) z = -z;
    D[i] = Dg[i];
    Z[i] = z;
  }
  __syncthreads();
  for (int i = tid; i < m; i += PT) {
    const double di = D[i];
    int rk = 0;
#pragma unroll 8
    for (int j = 0; j < m; ++j) {
      const double dj = D[j];
      rk += (dj < di) || (dj == di && j < i);
    }
    ds[rk] = di;
    zs[rk] = Z[i];
    pm[rk] = i;
  }
  __syncthreads();
  // the entries that z keeps move to the front, in order (one entry per thread)
  int *sel = reinterpret_cast<int *>(aux + AUX_SEL(n)) + r0;
  static_assert(PT >= DC_MAX, "one thread per entry");
  const int lane = tid & 63, wave = tid >> 6;
  const bool in = tid < m;
  const double ti = in ? ds[tid] : 0.0, zi = in ? zs[tid] : 0.0;
  double big = fabs(ti);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
  if (lane == 0) wred[wave] = big;
  __syncthreads();
  for (int w = 0; w < PT / 64; ++w) big = fmax(big, wred[w]);
  const double tol = 8.0 * DC_EPS * fmax(big, 0.25);
  const bool keep = in && rho * fabs(zi) > tol;
  const unsigned long long mask = __ballot(keep);
  if (lane == 0) wcnt[wave] = __popcll(mask);
  if (tid == 0) sh[1] = 0;
  __syncthreads();
  int before = __popcll(mask & ((1ull << lane) - 1)), kept = 0;
  for (int w = 0; w < PT / 64; ++w) {
    before += w < wave ? wcnt[w] : 0;
    kept += wcnt[w];
  }
  const int at = keep ? before : m - 1 - (tid - before);
  if (in) {
    D[at] = ti;
    Z[at] = zi;
    pk[at] = pm[tid];
  }
  if (tid == 0) sh[0] = kept;
  __syncthreads();
  if (tid + 1 < kept && near_pair(D[tid], Z[tid], D[tid + 1], Z[tid + 1], tol)) sh[1] = 1;
  __syncthreads();
  if (sh[1]) {  // uniform: the walk reads copies
    if (tid < kept) {
      ds[tid] = D[tid];
      zs[tid] = Z[tid];
      pm[tid] = pk[tid];
    }
    __syncthreads();
    if (tid == 0) {
      int nr;
      sh[0] = deflate(kept, tol, ds, zs, pm, D, Z, pk,
                      [&](int t, int a, int b, double c, double s) {
                        rp[t] = a;
                        rq[t] = b;
                        rc[t] = c;
                        rs[t] = s;
                      },
                      nr);
      sh[1] = nr;
    }
  }
  __syncthreads();
  const int k = sh[0], nr = sh[1];
  double *gd = aux + AUX_DS(n) + r0, *gz = aux + AUX_ZS(n) + r0, *dn = aux + AUX_D(n, par ^ 1) + r0;
  if (tid == 0) reinterpret_cast<int *>(aux + AUX_K(n))[r0] = k;
  if (in) {
    gd[tid] = D[tid];
    sel[tid] = pk[tid];
    if (tid < k)
      gz[tid] = Z[tid];
    else
      dn[tid] = D[tid];  // deflated eigenvalues are final at this level
  }
  // rotations: a row per thread; a rotation's second column is usually the
  // next one's first, so its value stays in a register
  for (int i = tid; i < m; i += PT) {
    double carry = 0.0;
    int held = -1;
    double nb = nr > 0 ? Q[size_t(rq[0]) * n + i] : 0.0;
    for (int t = 0; t < nr; ++t) {
      const int a = rp[t], b = rq[t];
      if (held != a) {
        if (held >= 0) Q[size_t(held) * n + i] = carry;
        carry = Q[size_t(a) * n + i];
      }
      const double qb = nb;
      if (t + 1 < nr) nb = Q[size_t(rq[t + 1]) * n + i];
      const double c = rc[t], s = rs[t];
      Q[size_t(a) * n + i] = c * carry + s * qb;
      carry = c * qb - s * carry;
      held = b;
    }
    if (held >= 0) Q[size_t(held) * n + i] = carry;
  }
}

// roots: one wave each, poles over the lanes; blocks[b] = (task, node), y = chunk of 4 roots
template <int RA>
__device__ __forceinline__ void roots_run(int j, int k, double rho, const double *gd, const double *gz, const double *dl,
                                          double *DLc, double *dn) {
  const int lane = threadIdx.x & 63;
  double d[RA], w[RA];
  double wt = 0.0;
#pragma unroll
  for (int a = 0; a < RA; ++a) {
    const int i = lane + 64 * a;
    d[a] = i < k ? gd[i] : 4.0;  // no pole: away from every root, weight 0
    const double z = i < k ? gz[i] : 0.0;
    w[a] = rho * z * z;
    wt += w[a];
  }
  wt = wave_total(wt);
  int K;
  double mu;
  auto sums = [&](double dK, double mu2) {
    SecSums s{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int a = 0; a < RA; ++a) secular_term((d[a] - dK) - mu2, w[a], s);
    double y[4] = {s.p, s.pp, s.f, s.fp};
    const double t = wave_totals<4>(y);
    return SecSums{read_lane(t, 0), read_lane(t, 16), read_lane(t, 32), read_lane(t, 48)};
  };
  secular_root(j, k, dl, wt, [&](int a) { return rho * gz[a] * gz[a]; }, sums, K, mu);
  const double dK = dl[K];
#pragma unroll
  for (int a = 0; a < RA; ++a) {
    const int i = lane + 64 * a;
    if (i < k) DLc[i] = (d[a] - dK) - mu;
  }
  if (lane == 0) dn[j] = dK + mu;
}

__global__ __launch_bounds__(256) void k_dc_roots(const DcTask *__restrict__ tasks, const int2 *__restrict__ blocks,
                                                  double *__restrict__ W, int l) {
  __shared__ double dl[DC_MAX];
  const int2 bk = blocks[blockIdx.x];
  const DcTask tk = tasks[bk.x];
  const int n = tk.n, p = tk.p, par = (l - 7) & 1;
  const int r0 = node_row(bk.y, l, n, p), md = node_row(2 * bk.y + 1, l - 1, n, p);
  double *aux = W + tk.x_off;
  const int k = reinterpret_cast<const int *>(aux + AUX_K(n))[r0];
  const int j0 = blockIdx.y * 4;
  if (j0 >= k) return;
  const double *gd = aux + AUX_DS(n) + r0, *gz = aux + AUX_ZS(n) + r0;
  for (int i = threadIdx.x; i < k; i += 256) dl[i] = gd[i];
  __syncthreads();
  const int j = j0 + (threadIdx.x >> 6);
  if (j >= k) return;  // no barrier below
  const double rho = 2.0 * fabs(W[tk.d_off + n + md - 1] / aux[AUX_SCALE(n)]);
  double *DLc = W + tk.q_off + 2 * size_t(n) * n + size_t(r0 + j) * n + r0, *dn = aux + AUX_D(n, par ^ 1) + r0;
  if (k <= 128)
    roots_run<2>(j, k, rho, gd, gz, dl, DLc, dn);
  else if (k <= 256)
    roots_run<4>(j, k, rho, gd, gz, dl, DLc, dn);
  else
    roots_run<8>(j, k, rho, gd, gz, dl, DLc, dn);
}

// vectors of the secular problem: every workgroup forms the whole z (its
// product over the roots split over the threads), then 64 columns
constexpr int VT = 1024, VC = 64;
__global__ __launch_bounds__(VT) void k_dc_vecs(const DcTask *__restrict__ tasks, const int2 *__restrict__ blocks,
                                                double *__restrict__ W, int l) {
  __shared__ double dl[DC_MAX], zh[DC_MAX], part[VT];
  const int2 bk = blocks[blockIdx.x];
  const DcTask tk = tasks[bk.x];
  const int n = tk.n, p = tk.p, tid = threadIdx.x;
  const int r0 = node_row(bk.y, l, n, p);
  double *aux = W + tk.x_off;
  const int k = reinterpret_cast<const int *>(aux + AUX_K(n))[r0];
  const int c0 = blockIdx.y * VC;
  if (c0 >= k) return;
  const double *gd = aux + AUX_DS(n) + r0, *gz = aux + AUX_ZS(n) + r0;
  double *DL = W + tk.q_off + 2 * size_t(n) * n + size_t(r0) * n + r0, *ZN = W + tk.q_off + 3 * size_t(n) * n +
                                                                            size_t(r0) * n + r0;
  for (int i = tid; i < k; i += VT) dl[i] = gd[i];
  __syncthreads();
  const int kp = (k + 63) & ~63, np = VT / kp;  // rows padded to waves, parts of the product
  {
    const int i = tid % kp, q = tid / kp;
    double pr = 1.0;
    if (q < np && i < k) {
      const double di = dl[i];
      const int per = (k + np - 1) / np, a1 = min(k, (q + 1) * per);
#pragma unroll 4
      for (int a = q * per; a < a1; ++a) {
        const double del = DL[size_t(a) * n + i];
        pr *= a == i ? -del : del * fast_rcp(di - dl[a]);
      }
    }
    part[tid] = pr;
  }
  __syncthreads();
  for (int i = tid; i < k; i += VT) {
    double pr = 1.0;
    for (int q = 0; q < np; ++q) pr *= part[q * kp + i];
    zh[i] = copysign(sqrt(fmax(pr, 0.0)), gz[i]);
  }
  __syncthreads();
  const int lane = tid & 63, wave = tid >> 6;
  for (int c = c0 + wave; c < min(k, c0 + VC); c += VT / 64) {
    const double *src = DL + size_t(c) * n;
    double v[DC_MAX / 64], nn = 0.0;
#pragma unroll
    for (int a = 0; a < DC_MAX / 64; ++a) {
      const int i = lane + 64 * a;
      v[a] = i < k ? zh[i] * fast_rcp(src[i]) : 0.0;
      nn += v[a] * v[a];
    }
    const double f = fast_rsqrt(wave_total(nn));
#pragma unroll
    for (int a = 0; a < DC_MAX / 64; ++a) {
      const int i = lane + 64 * a;
      if (i < k) ZN[size_t(c) * n + i] = v[a] * f;
    }
  }
}

// Qn(:, c) = sum_l Qo(:, sel(l)) S(l, c) for c < k, the deflated columns
// copied: 64 x 64 tiles, four waves of 16 columns, 16-deep stages in LDS
constexpr int GT = 64, GK = 16;
__global__ __launch_bounds__(256) void k_dc_product(const DcTask *__restrict__ tasks, const int2 *__restrict__ blocks,
                                                    double *__restrict__ W, int l) {
  __shared__ double As[2][GK * (GT + 4)], Bs[2][GT * (GK + 1)];
  const int2 bk = blocks[blockIdx.x];
  const DcTask tk = tasks[bk.x];
  const int n = tk.n, p = tk.p, par = (l - 7) & 1, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r0 = node_row(bk.y, l, n, p), m = node_row(bk.y + 1, l, n, p) - r0;
  const int mt = (m + GT - 1) / GT, tm = blockIdx.y % mt, tn = blockIdx.y / mt;
  if (tn >= mt) return;
  const double *aux = W + tk.x_off;
  const int k = reinterpret_cast<const int *>(aux + AUX_K(n))[r0];
  const int *sel = reinterpret_cast<const int *>(aux + AUX_SEL(n)) + r0;
  const size_t blk = size_t(r0) * n + r0, nn = size_t(n) * n;
  const double *Qo = W + tk.q_off + (par ? nn : 0) + blk;
  double *Qn = W + tk.q_off + (par ? 0 : nn) + blk;
  const double *S = W + tk.q_off + 3 * nn + blk;
  const int m0 = tm * GT, c0 = tn * GT;
  if (c0 < k) {
    typedef double v4 __attribute__((ext_vector_type(4)));
    v4 acc[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) acc[a] = v4{0, 0, 0, 0};
    double ra[4], rb[4];
    // A: row lane, k = wave + 4 u; B: k = tid % 16, column tid / 16 + 16 u
    auto load = [&](int l0) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int ka = l0 + wave + 4 * u, row = m0 + lane;
        ra[u] = (ka < k && row < m) ? Qo[size_t(sel[ka < k ? ka : 0]) * n + row] : 0.0;
        const int kb = l0 + (tid & 15), c = c0 + (tid >> 4) + 16 * u;
        rb[u] = (kb < k && c < k) ? S[size_t(c) * n + kb] : 0.0;
      }
    };
    auto store = [&](int b) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        As[b][(wave + 4 * u) * (GT + 4) + lane] = ra[u];
        Bs[b][((tid >> 4) + 16 * u) * (GK + 1) + (tid & 15)] = rb[u];
      }
    };
    load(0);
    store(0);
    __syncthreads();
    int cur = 0;
    for (int l0 = 0; l0 < k; l0 += GK) {
      const bool more = l0 + GK < k;
      if (more) load(l0 + GK);
#pragma unroll
      for (int q = 0; q < GK / 4; ++q) {
        const int kr = 4 * q + (lane >> 4);
        const double b = Bs[cur][(16 * wave + (lane & 15)) * (GK + 1) + kr];
#pragma unroll
        for (int a = 0; a < 4; ++a)
          acc[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(b, As[cur][kr * (GT + 4) + 16 * a + (lane & 15)], acc[a], 0, 0, 0);
      }
      if (more) store(cur ^ 1);
      __syncthreads();
      cur ^= 1;
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = c0 + 16 * wave + (lane >> 4) + 4 * r, row = m0 + 16 * a + (lane & 15);
        if (c < k && row < m) Qn[size_t(c) * n + row] = acc[a][r];
      }
  }
  // deflated columns of this tile
  for (int c = max(k, c0) + wave; c < min(m, c0 + GT); c += 4) {
    const int row = m0 + lane;
    if (row < m) Qn[size_t(c) * n + row] = Qo[size_t(sel[c]) * n + row];
  }
}

__global__ void k_dc_zero(const DcTask *__restrict__ tasks, double *__restrict__ W) {
  const DcTask tk = tasks[blockIdx.x];
  const size_t e = 2 * size_t(tk.n) * tk.n;
  for (size_t x = size_t(blockIdx.y) * 256 + threadIdx.x; x < e; x += size_t(gridDim.y) * 256) W[tk.q_off + x] = 0.0;
}

// eigenvalues descending (equal ones in column order) to w and the host,
// and the column that each goes to; the last of `count` matrices raises the
// host's flag
__device__ __forceinline__ void rank_run(const DcTask &tk, int index, double *__restrict__ D, const DcOut &out,
                                         const double *__restrict__ W, double *__restrict__ wout) {
  const int n = tk.n, tid = threadIdx.x;
  const double *aux = W + tk.x_off;
  const double *Dg = aux + AUX_D(n, tk.p > 6 ? (tk.p - 6) & 1 : 0);
  const double scaled = aux[AUX_SCALE(n)], scale = scaled <= DBL_MAX ? scaled : 1.0;
  for (int i = tid; i < n; i += blockDim.x) D[i] = Dg[i];
  __syncthreads();
  for (int i = tid; i < n; i += blockDim.x) {
    const double di = D[i];
    int rk = 0;
#pragma unroll 8
    for (int j = 0; j < n; ++j) {
      const double dj = D[j];
      rk += (dj > di) || (dj == di && j < i);
    }
    out.rank[tk.r_off + i] = rk;
    wout[tk.w_off + rk] = di * scale;
    out.hw[tk.r_off + rk] = di * scale;
  }
  if (tid == 0) out.hstatus[index] = out.status[index];
  __threadfence_system();
  __syncthreads();
  if (tid == 0 && atomicAdd(out.done, 1u) == unsigned(out.count - 1)) {
    __threadfence_system();
    *reinterpret_cast<volatile unsigned long long *>(out.flag) = out.seq;
  }
}

// tasks first .. first + gridDim.x - 1
__global__ __launch_bounds__(PT) void k_dc_rank(const DcTask *__restrict__ tasks, int first, const double *__restrict__ W,
                                                double *__restrict__ wout, DcOut out) {
  __shared__ double D[DC_MAX];
  const DcTask tk = tasks[first + blockIdx.x];
  rank_run(tk, first + blockIdx.x, D, out, W, wout);
}

// ---- matrices of at most 64 rows: everything in one launch -------------------------
// Reduction, divide and conquer, ranks and back-transformation by the same
// workgroup: at this size a launch costs as much as a phase (density-matrix
// blocks of 30 rows: 15 + 30 + 5 + 5 us in four launches with the gaps
// between them).
__global__ __launch_bounds__(ST) void k_syev_small(const TriTask *__restrict__ tri, const DcTask *__restrict__ tasks,
                                                   const BackTask *__restrict__ back, double *__restrict__ A,
                                                   double *__restrict__ W, double *__restrict__ wout, DcOut out,
                                                   int first) {
  __shared__ __align__(16) double lds[tri_lds<1, false>()];
  __shared__ double D[SB];
  const int b = first + blockIdx.x;
  int *st = out.status + b;
  tri_run<1, false>(tri[b], 0, A, W, st, lds);
  __syncthreads();
  const DcTask tk = tasks[b];
  dc_small_run(tk, 0, W, st);
  __syncthreads();
  rank_run(tk, b, D, out, W, wout);
  __syncthreads();
  if (*st != 0) return;  // uniform
  const BackTask bt = back[b];
  for (int c = QCB * (threadIdx.x >> 6); c < tk.n; c += QCB * (ST / 64)) back_run<1, 4>(bt, c, W, W, A, out.rank);
}

}  // namespace

void dc_blocks(const std::vector<DcTask> &tasks, int ntasks, std::vector<int2> &blocks, std::vector<DcLevel> &levels) {
  int pmax = 0;
  for (int i = 0; i < ntasks; ++i) pmax = std::max(pmax, tasks[size_t(i)].p);
  for (int l = 6; l <= pmax; ++l) {
    DcLevel lv{l, blocks.size(), 0, 0};
    for (int i = 0; i < ntasks; ++i) {
      const DcTask &t = tasks[size_t(i)];
      if (t.p < l) continue;
      const int nodes = 1 << (t.p - l);
      for (int x = 0; x < nodes; ++x) blocks.push_back(make_int2(i, x));
      lv.maxm = std::max(lv.maxm, (t.n + nodes - 1) / nodes);
    }
    lv.count = blocks.size() - lv.first;
    levels.push_back(lv);
  }
}

void dc_launch(itx_ctx *ctx, const DcTask *tasks, int ntasks, const int2 *blocks, const std::vector<DcLevel> &levels,
               double *W, double *w, const DcOut &out) {
  const hipStream_t st = ctx->stream;
  if (ntasks == 0) return;
  hipLaunchKernelGGL(k_dc_zero, dim3(unsigned(ntasks), 32), dim3(256), 0, st, tasks, W);
  for (const DcLevel &lv : levels) {
    const unsigned nb = unsigned(lv.count);
    const int2 *b = blocks + lv.first;
    if (lv.level == 6) {
      hipLaunchKernelGGL(k_dc_small, dim3(nb), dim3(ST), 0, st, tasks, b, W, out.status);
      continue;
    }
    const unsigned m = unsigned(lv.maxm), mt = (m + GT - 1) / GT;
    hipLaunchKernelGGL(k_dc_prep, dim3(nb), dim3(PT), 0, st, tasks, b, W, lv.level);
    hipLaunchKernelGGL(k_dc_roots, dim3(nb, (m + 3) / 4), dim3(256), 0, st, tasks, b, W, lv.level);
    hipLaunchKernelGGL(k_dc_vecs, dim3(nb, (m + VC - 1) / VC), dim3(VT), 0, st, tasks, b, W, lv.level);
    // the eigenvalues are whole before the last product
    if (&lv == &levels.back())
      hipLaunchKernelGGL(k_dc_rank, dim3(unsigned(ntasks)), dim3(PT), 0, st, tasks, 0, W, w, out);
    hipLaunchKernelGGL(k_dc_product, dim3(nb, mt * mt), dim3(256), 0, st, tasks, b, W, lv.level);
  }
}

void syev_small_launch(itx_ctx *ctx, const TriTask *tri, const DcTask *tasks, const BackTask *back, int first, int count,
                       double *A, double *W, double *w, const DcOut &out) {
  if (count)
    hipLaunchKernelGGL(k_syev_small, dim3(unsigned(count)), dim3(ST), 0, ctx->stream, tri, tasks, back, A, W, w, out,
                       first);
}

}  // namespace itx
