// FP64 singular value decomposition of libitx (one workgroup per matrix).
//
// Replaces the SVD(M,U,D,V) call of svdImpl (svd.cc:87,206-213, through
// SVDRef, tensor/algs.cc:586-631, i.e. dgesdd or the density-matrix method
// of SVDRefImpl): A = U diag(S) V^T with S descending, U and V with
// orthonormal columns, for every block of a QN tensor in one launch.
//
// Method (textbook, not LAPACK's code): one-sided Jacobi (Hestenes, J. SIAM
// 6 (1958) 51).  The k = min(m,n) columns of X (X = A^T when m <= n, else
// A; columns of length max(m,n)) are rotated pairwise until every pair is
// orthogonal to a relative tolerance; the rotations accumulate in J.  Then
// the singular values are the column norms of X, the normalised columns
// of X are the singular vectors of the long side and J holds those of the
// short side.  One-sided Jacobi keeps the small singular values and their
// vectors accurate without the refinement step the density-matrix method
// needs.  Pairs are scheduled round-robin (k/2 disjoint pairs per round,
// k-1 rounds per sweep), each pair reduced by a group of lanes.
#include <algorithm>
#include <cfloat>
#include <cstring>
#include <type_traits>

#include "itx_eig.h"

namespace itx {
namespace {

constexpr int SVD_MAX_SWEEPS = 60;  // sweeps before reporting no convergence
// X and J in LDS (columns at odd pitches) when they fit, else in the workspace
constexpr size_t SVD_LDS = 160 * 1024 - 512;  // of 160 KB: 100 x 100 fits
__host__ __device__ inline size_t svd_lds(int m, int n) {
  const size_t R = m < n ? m : n, C = m < n ? n : m;
  return sizeof(double) * R * ((C | 1) + (R | 1));
}

struct SvdTask {
  int32_t m, n;
  int64_t a_off, u_off, s_off, v_off;
  int64_t x_off;  // workspace: X (C x R), J (R x R), sigma (R), rank (R)
};

// sums of three values over the G lanes of a group, step by step so that
// the three chains overlap
template <int G>
__device__ __forceinline__ void group_sums(double &a, double &b, double &c) {
  if constexpr (G > 1) a += dpp_move<DPP_XOR1>(a), b += dpp_move<DPP_XOR1>(b), c += dpp_move<DPP_XOR1>(c);
  if constexpr (G > 2) a += dpp_move<DPP_XOR2>(a), b += dpp_move<DPP_XOR2>(b), c += dpp_move<DPP_XOR2>(c);
  if constexpr (G > 4)
    a += dpp_move<DPP_HALF_MIRROR>(a), b += dpp_move<DPP_HALF_MIRROR>(b), c += dpp_move<DPP_HALF_MIRROR>(c);
  if constexpr (G > 8) a += dpp_move<DPP_ROR8>(a), b += dpp_move<DPP_ROR8>(b), c += dpp_move<DPP_ROR8>(c);
  if constexpr (G > 16) a = swap16_add(a, a), b = swap16_add(b, b), c = swap16_add(c, c);
  if constexpr (G > 32) a = swap32_add(a, a), b = swap32_add(b, b), c = swap32_add(c, c);
}

// One workgroup per matrix.  A sweep is R - 1 dependent rounds of R / 2
// independent pairs, so a round's latency bounds it: a pair has up to 64
// lanes, its columns come from LDS where the matrix fits, and a barrier
// orders LDS only (blocks up to 37 x 37: 0.42 ms for some 10 sweeps, 1.1 us
// a round; from the workspace, with 256 threads, 1.14 ms).  ST: threads per
// matrix, 1024 or, for large batches of small matrices, 256.
template <int ST, bool LDS, int G>
__device__ __forceinline__ void gesvd_run(const SvdTask &tk, const double *__restrict__ Abase,
                                          double *__restrict__ Ubase, double *__restrict__ Sbase,
                                          double *__restrict__ Vbase, double *__restrict__ Wbase,
                                          int *__restrict__ status, double *lds, int *sh_rot) {
  const int m = tk.m, n = tk.n;
  const int R = min(m, n), C = max(m, n);
  const int tid = threadIdx.x;
  const double *__restrict__ A = Abase + tk.a_off;
  const int PX = LDS ? (C | 1) : C, PJ = LDS ? (R | 1) : R;  // column pitches
  double *X = LDS ? lds : Wbase + tk.x_off;
  double *J = X + size_t(PX) * R;
  double *__restrict__ sig = Wbase + tk.x_off + (LDS ? 0 : size_t(C) * R + size_t(R) * R);
  double *__restrict__ rnk = sig + R;
  const bool wide = m <= n;  // X = A^T
  auto meet = [&]() {
    if constexpr (LDS)
      lds_barrier();
    else
      __syncthreads();
  };

  using Count = std::conditional_t<LDS, int, size_t>;
  const Count cr = Count(C) * R, rr = Count(R) * R;
  for (Count x = tid; x < cr; x += ST) {  // A read in its own order
    const Count i = x % m, j = x / m;
    (wide ? X[size_t(i) * PX + j] : X[size_t(j) * PX + i]) = A[x];
  }
  for (Count x = tid; x < rr; x += ST) J[size_t(x / R) * PJ + x % R] = (x % R == x / R) ? 1.0 : 0.0;
  if (tid < 2) sh_rot[tid] = 0;
  __syncthreads();

  // round-robin schedule over Rp (even) slots; slot R is a dummy when R is odd
  const int Rp = R + (R & 1), P = Rp / 2;
  const int NG = ST / G, grp = tid / G, g = tid % G;
  const double tol = 4.0 * DBL_EPSILON * sqrt(double(C));

  int sweep = 0;
  for (; sweep < SVD_MAX_SWEEPS; ++sweep) {
    for (int k = 0; k < Rp - 1; ++k) {
      for (int p = grp; p < P; p += NG) {
        auto pos = [&](int x) {
          const int y = x - 1 + k;
          return x == 0 ? 0 : 1 + (y >= Rp - 1 ? y - (Rp - 1) : y);
        };
        int a = pos(p), b = pos(Rp - 1 - p);
        if (a >= R || b >= R) continue;  // group-uniform
        if (a > b) {
          const int t = a;
          a = b;
          b = t;
        }
        double *xa = X + size_t(a) * PX, *xb = X + size_t(b) * PX;
        double *ja = J + size_t(a) * PJ, *jb = J + size_t(b) * PJ;
        // the first four elements of a lane stay in registers from the sums
        // to the rotation, and J's are on their way meanwhile
        double xu[4], xv[4], ju[4], jv[4];
        double al = 0, be = 0, ga = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int c = g + G * t;
          xu[t] = c < C ? xa[c] : 0.0;
          xv[t] = c < C ? xb[c] : 0.0;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int c = g + G * t;
          ju[t] = c < R ? ja[c] : 0.0;
          jv[t] = c < R ? jb[c] : 0.0;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          al = fma(xu[t], xu[t], al);
          be = fma(xv[t], xv[t], be);
          ga = fma(xu[t], xv[t], ga);
        }
#pragma unroll 2
        for (int c = g + 4 * G; c < C; c += G) {
          const double u = xa[c], v = xb[c];
          al = fma(u, u, al);
          be = fma(v, v, be);
          ga = fma(u, v, ga);
        }
        group_sums<G>(al, be, ga);
        // rotate unless the pair is orthogonal to working precision; the
        // products of the fast form stay in range for norms within 1e+-35
        double cs, sn;
        const double top = fmax(al, be), low = fmin(al, be);
        if (top < 1e70 && low > 1e-70) {
          if (ga * ga <= tol * tol * (al * be)) continue;
          // t = tan of the angle that zeroes ga: the smaller root of t^2 + 2 zeta t - 1
          const double dl = be - al, g2 = 2.0 * ga;
          const double t = copysign(g2, dl >= 0.0 ? ga : -ga) * fast_rcp(fabs(dl) + fast_sqrt(fma(dl, dl, g2 * g2)));
          cs = fast_rsqrt(fma(t, t, 1.0));
          sn = cs * t;
        } else {
          if (ga == 0.0 || al == 0.0 || be == 0.0 || fabs(ga) <= tol * sqrt(al) * sqrt(be)) continue;
          // What is left of a column that depends on the others shrinks from sweep
          // to sweep (where rows repeat, by 1e6), and once its square is denormal
          // no rotation makes it orthogonal to working precision.  Then, or past
          // the sweeps that independent columns take, it is zero beside a column
          // more than 1e30 times as long.
          if ((low < 1e-290 && top > 1e-230) || (sweep >= 20 && low < 1e-60 * top)) {
            double *x = al < be ? xa : xb;
            for (int c = g; c < C; c += G) x[c] = 0.0;
            continue;
          }
          const double zeta = (be - al) / (2.0 * ga), z = fabs(zeta);
          const double t = copysign(1.0, zeta) / (z + (z < 1e150 ? sqrt(fma(z, z, 1.0)) : z));
          if (t == 0.0) continue;  // past the smallest number
          cs = 1.0 / sqrt(fma(t, t, 1.0));
          sn = cs * t;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int c = g + G * t;
          if (c < C) {
            xa[c] = cs * xu[t] - sn * xv[t];
            xb[c] = sn * xu[t] + cs * xv[t];
          }
          if (c < R) {
            ja[c] = cs * ju[t] - sn * jv[t];
            jb[c] = sn * ju[t] + cs * jv[t];
          }
        }
#pragma unroll 2
        for (int c = g + 4 * G; c < C; c += G) {
          const double u = xa[c], v = xb[c];
          xa[c] = cs * u - sn * v;
          xb[c] = sn * u + cs * v;
        }
#pragma unroll 2
        for (int r = g + 4 * G; r < R; r += G) {
          const double u = ja[r], v = jb[r];
          ja[r] = cs * u - sn * v;
          jb[r] = sn * u + cs * v;
        }
        if (g == 0) sh_rot[sweep & 1] = 1;
      }
      meet();
    }
    // this sweep's flag was set before the round's barrier; the other one is
    // cleared for the next sweep, whose rounds begin after the barrier below
    const int rot = sh_rot[sweep & 1];
    if (tid == 0) sh_rot[(sweep + 1) & 1] = 0;
    meet();
    if (!rot) break;
  }
  if (sweep == SVD_MAX_SWEEPS) {
    if (tid == 0) *status = 1;
    return;
  }

  // singular values (column norms) and their descending stable ranks
  for (int r = grp; r < R; r += NG) {
    const double *xr = X + size_t(r) * PX;
    double s = 0;
    for (int c = g; c < C; c += G) s = fma(xr[c], xr[c], s);
    double o1 = 0, o2 = 0;
    group_sums<G>(s, o1, o2);
    if (g == 0) sig[r] = sqrt(s);
  }
  __syncthreads();
  for (int r = tid; r < R; r += ST) {
    const double sr = sig[r];
    int rank = 0;
#pragma unroll 4
    for (int j = 0; j < R; ++j) rank += (sig[j] > sr) || (sig[j] == sr && j < r);
    rnk[r] = double(rank);
  }
  __syncthreads();
  double *__restrict__ U = Ubase + tk.u_off;
  double *__restrict__ V = Vbase + tk.v_off;
  double *__restrict__ S = Sbase + tk.s_off;
  double *__restrict__ Long = wide ? V : U;    // C x R: normalised columns of X
  double *__restrict__ Short = wide ? U : V;   // R x R: J
  for (int r = tid; r < R; r += ST) S[int(rnk[r])] = sig[r];
  for (Count x = tid; x < cr; x += ST) {
    const Count c = x % C, r = x / C;
    const double sr = sig[r];
    Long[size_t(rnk[r]) * C + c] = sr > 0.0 ? X[size_t(r) * PX + c] / sr : 0.0;
  }
  for (Count x = tid; x < rr; x += ST) {
    const Count i = x % R, r = x / R;
    Short[size_t(rnk[r]) * R + i] = J[size_t(r) * PJ + i];
  }
  if (tid == 0) *status = 0;
}

template <int ST>
__global__ __launch_bounds__(ST) void k_gesvd(const SvdTask *__restrict__ tasks, const double *__restrict__ Abase,
                                              double *__restrict__ Ubase, double *__restrict__ Sbase,
                                              double *__restrict__ Vbase, double *__restrict__ Wbase,
                                              int *__restrict__ status, unsigned lds_bytes) {
  extern __shared__ double lds[];
  __shared__ int sh_rot[2];
  const SvdTask tk = tasks[blockIdx.x];
  int *st = status + blockIdx.x;
  if (min(tk.m, tk.n) <= 0) {
    if (threadIdx.x == 0) *st = 0;
    return;
  }
  // as many lanes per pair as the threads allow for all pairs of a round
  const int P = (min(tk.m, tk.n) + 1) / 2;
#define ITX_SVD(L, G) gesvd_run<ST, L, G>(tk, Abase, Ubase, Sbase, Vbase, Wbase, st, lds, sh_rot)
  if constexpr (ST == 256) {  // at most 64 rows and columns, in LDS
    if (P * 64 <= ST)
      ITX_SVD(true, 64);
    else if (P * 32 <= ST)
      ITX_SVD(true, 32);
    else if (P * 16 <= ST)
      ITX_SVD(true, 16);
    else
      ITX_SVD(true, 8);
  } else {
    const bool in = svd_lds(tk.m, tk.n) <= lds_bytes;
    if (in && P * 64 <= ST)
      ITX_SVD(true, 64);
    else if (in && P * 32 <= ST)
      ITX_SVD(true, 32);
    else if (in)  // at most 51 pairs fit
      ITX_SVD(true, 16);
    else if (P * 64 <= ST)
      ITX_SVD(false, 64);
    else if (P * 16 <= ST)
      ITX_SVD(false, 16);
    else if (P * 4 <= ST)
      ITX_SVD(false, 4);
    else
      ITX_SVD(false, 1);
  }
#undef ITX_SVD
}

}  // namespace
}  // namespace itx

extern "C" int itx_gesvd_batched(itx_ctx *ctx, int nmat, const int32_t *m, const int32_t *n, const int64_t *a_offs,
                                 const double *A, const int64_t *u_offs, double *U, const int64_t *s_offs, double *S,
                                 const int64_t *v_offs, double *V) {
  if (!ctx || nmat < 0 || (nmat > 0 && (!m || !n || !a_offs || !u_offs || !s_offs || !v_offs))) return ITX_ERR_ARG;
  if (nmat == 0) return ITX_OK;
  std::vector<itx::SvdTask> tasks(static_cast<size_t>(nmat));
  int64_t wsize = 0;
  for (int b = 0; b < nmat; ++b) {
    if (m[b] < 0 || n[b] < 0) return itx::set_err(ctx, ITX_ERR_ARG, "itx_gesvd: negative dimension");
    const int64_t R = std::min(m[b], n[b]), C = std::max(m[b], n[b]);
    auto &t = tasks[size_t(b)];
    t.m = m[b];
    t.n = n[b];
    t.a_off = a_offs[b];
    t.u_off = u_offs[b];
    t.s_off = s_offs[b];
    t.v_off = v_offs[b];
    t.x_off = wsize;
    wsize += C * R + R * R + 2 * R;
  }
  // A CU holds one workgroup of 1024 threads (83 registers) and five of 256:
  // more small matrices than CUs take 256.  30 x 30 x 600 1.19 to 0.36 ms (four
  // waves over the workspace took 0.85), 8 x 8 x 4000 0.77 to 0.45, 64 x 64 x
  // 300 1.86 to 1.44; above 64 rows or columns it loses (80 x 80 x 512 2.9 to 5.6).
  auto is_large = [](const itx::SvdTask &t) { return std::max(t.m, t.n) > 64; };
  int nlarge = int(std::count_if(tasks.begin(), tasks.end(), is_large));
  if (nmat - nlarge > ctx->num_cus)
    std::stable_partition(tasks.begin(), tasks.end(), is_large);
  else
    nlarge = nmat;
  const size_t tbytes = sizeof(itx::SvdTask) * size_t(nmat), sbytes = sizeof(int) * size_t(nmat);
  const size_t woff = (tbytes + sbytes + 255) & ~size_t(255);
  void *ws = nullptr;
  int rc = itx::pool_alloc(ctx, woff + sizeof(double) * size_t(std::max<int64_t>(wsize, 1)), &ws);
  if (rc) return rc;
  char *wsb = static_cast<char *>(ws);
  rc = itx::stage_upload(ctx, wsb, tasks.data(), tbytes);
  if (rc) {
    itx::pool_free(ctx, ws);
    return rc;
  }
  int *dst = reinterpret_cast<int *>(wsb + tbytes);
  // large matrices first, 1024 threads each, then the small ones
  for (int part = 0; part < 2; ++part) {
    const int first = part ? nlarge : 0, count = part ? nmat - nlarge : nlarge;
    if (!count) continue;
    size_t lds = 0;  // for the largest matrix that fits
    for (int b = first; b < first + count; ++b) {
      const size_t need = itx::svd_lds(tasks[size_t(b)].m, tasks[size_t(b)].n);
      if (need <= itx::SVD_LDS) lds = std::max(lds, need);
    }
    hipLaunchKernelGGL(part ? itx::k_gesvd<256> : itx::k_gesvd<1024>, dim3(unsigned(count)), dim3(part ? 256 : 1024), lds,
                       ctx->stream, reinterpret_cast<const itx::SvdTask *>(wsb) + first, A, U, S, V,
                       reinterpret_cast<double *>(wsb + woff), dst + first, unsigned(lds));
  }
  hipError_t e = hipGetLastError();
  std::vector<int> st(static_cast<size_t>(nmat), 0);
  if (e == hipSuccess) e = hipMemcpyAsync(st.data(), dst, sbytes, hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  itx::pool_free(ctx, ws);
  if (e != hipSuccess) return itx::hip_err(ctx, e, "itx_gesvd");
  for (int b = 0; b < nmat; ++b)
    if (st[size_t(b)] != 0) return itx::set_err(ctx, ITX_ERR_NOCONV, "itx_gesvd: Jacobi sweeps did not converge");
  return ITX_OK;
}

extern "C" int itx_gesvd(itx_ctx *ctx, int m, int n, const double *A, double *U, double *S, double *V) {
  if (!ctx || m < 0 || n < 0) return ITX_ERR_ARG;
  const int32_t mm[1] = {m}, nn[1] = {n};
  const int64_t z[1] = {0};
  return itx_gesvd_batched(ctx, 1, mm, nn, z, A, z, U, z, S, z, V);
}
