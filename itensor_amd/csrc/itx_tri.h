// Device code of the Householder reduction and of the products with its
// orthogonal factor, shared by the kernels of itx_tridiag.hip (any order)
// and the one-launch kernel of itx_dc.hip (at most 64 rows).  Textbook
// Householder reduction; Golub & Van Loan, "Matrix Computations", 8.3.
#pragma once

#include <cfloat>

#include "itx_eig.h"

namespace itx {
namespace {

// ---- reduction --------------------------------------------------------------
// The matrix lives in registers for the whole reduction.  A Householder step
// k needs one meeting of the waves:
//   - every thread applies the pending rank-2 update of step k-1 to its
//     elements and forms its part of p = tau S v_k;
//   - p and column k+1 are published, all waves meet, and each wave by
//     itself forms w_k = p - (tau/2 v.p) v, brings column k+1 up to date
//     and forms the reflector of step k+1 from it (lanes over rows).
// Up to 128 rows one workgroup of four waves holds the matrix (one wave per
// SIMD: the redundant reflector arithmetic of more waves would share the
// SIMDs), its 256 threads as a 16 x 16 grid over rows and columns: a thread
// then reads the pending (v, w) of 4 or 8 rows and columns (with whole
// columns per wave, three values for every column, a step at n = 64 took
// 1.65 us).  A step is one LDS round and one barrier.  Above, a wave
// owns whole columns (w, w + W, w + 2W, ... of the W waves of a matrix, lanes
// over rows), so that p_j = tau column_j . v_k needs no sum across waves,
// and workgroups of four waves with four columns each share a matrix and
// meet in global memory: every value has its own place per step, filled with
// a mark before the launch, and a reader polls the value itself until the
// mark is gone -- one trip through memory instead of data, flag and data
// again.  All values go through agent-scope atomics.  A wait is bounded: a
// lane that gives up sets the matrix's status and a mark of its workgroup, the
// waiting lanes of other workgroups look at the status now and then, and a
// workgroup that is marked runs to the end without waiting again, so that a
// workgroup that never runs costs one bound and not one per step.  The host
// then takes another path.
// What bounds it is the latency of the n - 2 dependent steps: in one
// workgroup 1.15 us a step at n = 64 and 1.6 at 128 (72 and 203 us in all;
// the LDS-resident form before this one 174 and 519), across workgroups 2.5
// us at n = 234, 1.3 of them the trip through memory (0.59 ms; one workgroup
// over the L2 2.7 ms).  Four columns per wave: with eight, on half the
// workgroups, the update costs what the trip gains.
constexpr int TNW = 4;            // waves per workgroup
constexpr int TNT = 64 * TNW;
constexpr int TXC = 4;            // columns per wave across workgroups
constexpr unsigned long long TRI_MARK = 0x7FF8DEADBEEF4242ull;  // a quiet NaN no arithmetic makes
constexpr int TRI_LOOK = 1024;  // polls between looks at the status

template <int RA, bool MULTI>
constexpr int tri_lds() {  // doubles: per wave v, (v, w); twice p and column
  return (3 * TNW + 2 * (MULTI ? 2 : TNW + 1)) * 64 * RA;
}

template <int RA, bool MULTI>
__device__ __forceinline__ void tri_run(const TriTask &tk, int g, const double *__restrict__ Abase,
                                        double *__restrict__ W, int *__restrict__ status, double *__restrict__ lds,
                                        int polls = 0, int *gave = nullptr) {
  constexpr int NR = 64 * RA;
  // rows and columns of the matrix that a thread holds
  constexpr int XR = MULTI ? RA : 4 * RA, XC = MULTI ? TXC : 4 * RA;
  const int n = tk.n, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int NWV = MULTI ? tk.wgs * TNW : TNW, gw = MULTI ? g * TNW + wave : wave;
  const double *__restrict__ A = Abase + tk.a_off;
  double *__restrict__ V = W + tk.v_off;
  double *__restrict__ dv = W + tk.d_off, *__restrict__ ev = dv + n, *__restrict__ tv = ev + n;
  unsigned long long *ex = reinterpret_cast<unsigned long long *>(W + tk.x_off);
  if (n <= 2) {
    if (gw == 0 && lane == 0) {
      dv[0] = A[0];
      ev[0] = n == 2 ? A[1] : 0.0;
      if (n == 2) {
        dv[1] = A[3];
        ev[1] = 0.0;
      }
    }
    return;
  }
  // the wave's own copies: v of this step, (v, w) of the pending update
  double *lv = lds + wave * NR;
  double2 *lp = reinterpret_cast<double2 *>(lds + (TNW + 2 * wave) * NR);
  // published values, two sets by step parity: p (one workgroup: the waves'
  // partial sums of it) and a column
  constexpr int PP = MULTI ? 1 : TNW;
  double *sp = lds + 3 * TNW * NR, *sc = sp + 2 * PP * NR;

  // thread's rows ri + rd a and columns ci + cd s
  const int ri = MULTI ? lane : tid & 15, ci = MULTI ? gw : tid >> 4;
  const int rd = MULTI ? 64 : 16, cd = MULTI ? NWV : 16;
  double x[XC][XR];
#pragma unroll
  for (int s = 0; s < XC; ++s) {
    const int j = ci + cd * s;
#pragma unroll
    for (int a = 0; a < XR; ++a) {
      const int i = ri + rd * a;
      x[s][a] = (i < n && j < n) ? A[size_t(j) * n + i] : 0.0;
    }
  }
  double v[RA], wp[RA], c[RA], vp[RA];
  double tau = 0.0, al = 0.0;
  // element i (wave-uniform) of a vector held over the lanes
  auto pick = [&](const double(&u)[RA], int i) __attribute__((always_inline)) {
    double r = read_lane(u[0], i & 63);
#pragma unroll
    for (int a = 1; a < RA; ++a) {
      const double t = read_lane(u[a], i & 63);
      r = (i >> 6) == a ? t : r;
    }
    return r;
  };
  // the reflector of column q (rows > q + 1 of c and x0 = c[q + 1]), the same
  // in every wave; v in units of the column, a power of two, so that products
  // with much larger columns stay numbers
  auto reflect = [&](int q, double x0) __attribute__((always_inline)) {
    double sg = 0.0;
#pragma unroll
    for (int a = 0; a < RA; ++a)
      if (lane + 64 * a > q + 1) sg += c[a] * c[a];
    sg = wave_total(sg);
    double alpha = x0, v0 = x0;
    tau = 0.0;
    const double s2 = x0 * x0 + sg;
    // scalar branches: the slow forms are otherwise computed beside the fast ones
    if (__builtin_amdgcn_readfirstlane(s2 > 1e-280 && s2 < 1e280)) {
      if (__builtin_amdgcn_readfirstlane(sg > 0.0)) {
        const int ex = __builtin_amdgcn_frexp_exp(s2) >> 1;
        const double x = ldexp(x0, -ex), ss = ldexp(sg, -2 * ex), mu = fast_sqrt(ldexp(s2, -2 * ex));
        v0 = (x <= 0) ? x - mu : x + mu;
        alpha = ldexp((x <= 0) ? mu : -mu, ex);
#pragma unroll
        for (int a = 0; a < RA; ++a) c[a] = ldexp(c[a], -ex);
        tau = 2.0 * fast_rcp(v0 * v0 + ss);
      }
    } else if (sg != sg) {
      tau = sg;  // not a number: carried into d and e
    } else {
      // The squares leave the range of numbers, as in the last columns of a
      // matrix whose rank is small or whose rows are graded.
      double m = fabs(x0);
#pragma unroll
      for (int a = 0; a < RA; ++a)
        if (lane + 64 * a > q + 1) m = fmax(m, fabs(c[a]));
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
      if (m > DBL_MAX) {
        alpha = (x0 <= 0) ? m : -m;
      } else if (m > 0.0) {
        int ex;
        (void)frexp(m, &ex);
        sg = 0.0;
#pragma unroll
        for (int a = 0; a < RA; ++a) {
          c[a] = ldexp(c[a], -ex);
          if (lane + 64 * a > q + 1) sg += c[a] * c[a];
        }
        sg = wave_total(sg);
        if (sg > 0.0) {
          const double x = ldexp(x0, -ex), mu = sqrt(x * x + sg);
          v0 = (x <= 0) ? x - mu : x + mu;
          alpha = ldexp((x <= 0) ? mu : -mu, ex);
          tau = 2.0 / (v0 * v0 + sg);
        }
      }
    }
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const int i = lane + 64 * a;
      v[a] = (i <= q || tau == 0.0) ? 0.0 : (i == q + 1) ? v0 : c[a];
      lv[i] = v[a];
    }
    al = alpha;
  };
#pragma unroll
  for (int a = 0; a < RA; ++a) {
    const int i = lane + 64 * a;
    c[a] = i < n ? A[i] : 0.0;
    vp[a] = wp[a] = 0.0;
    lp[i] = make_double2(0.0, 0.0);
  }
  if (gw == 0 && lane == 0) dv[0] = A[0];
  reflect(0, A[1]);
  bool dead = false;
  int qw = MULTI ? 1 : 0, qs = 0;  // the wave and slot of column k + 1

  for (int k = 0; k + 2 < n; ++k) {
    // the wave's own LDS copies are ordered by the wave itself
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int par = k & 1;
    double *spk = sp + par * PP * NR, *sck = sc + par * NR;
    double y[MULTI ? XC : XR];
    double2 pc[XC];
#pragma unroll
    for (int s = 0; s < XC; ++s) pc[s] = lp[ci + cd * s];
    if constexpr (MULTI) {
#pragma unroll
      for (int s = 0; s < XC; ++s) {
        const int j = ci + cd * s;
        y[s] = 0.0;
        if (j > k && j < n) {  // wave-uniform
#pragma unroll
          for (int a = 0; a < RA; ++a) {
            x[s][a] = fma(-wp[a], pc[s].x, fma(-vp[a], pc[s].y, x[s][a]));
            y[s] += x[s][a] * v[a];
          }
        }
      }
    } else {
      double vc[XC];
#pragma unroll
      for (int s = 0; s < XC; ++s) vc[s] = lv[ci + cd * s];
#pragma unroll
      for (int a = 0; a < XR; ++a) {
        y[a] = 0.0;
        if (rd * a + 15 > k) {  // rows up to k take no further part
          const double2 pr = lp[ri + rd * a];
#pragma unroll
          for (int s = 0; s < XC; ++s) {
            x[s][a] = fma(-pr.y, pc[s].x, fma(-pr.x, pc[s].y, x[s][a]));
            y[a] += x[s][a] * vc[s];
          }
        }
      }
    }
    unsigned long long *exk = ex + size_t(k) * 2 * n;
    auto publish = [&](bool col, int i, double val) __attribute__((always_inline)) {
      if constexpr (MULTI) {
        unsigned long long b = (unsigned long long)__double_as_longlong(val);
        if (b == TRI_MARK) b ^= 1;
        __hip_atomic_store(exk + (col ? n : 0) + i, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        (void)col;
        (void)i;
        (void)val;
      }
    };
    const int q = k + 1;
    if constexpr (MULTI) {
      const double yt = wave_totals<XC>(y);
      const double pj = tau != 0.0 ? tau * yt : 0.0;  // no reflector: also beside infinite entries
      if (lane % (64 / XC) == 0) {
        const int j = ci + cd * (lane / (64 / XC));
        if (j > k && j < n) publish(false, j, pj);
      }
      if (qw == gw) {
#pragma unroll
        for (int s = 0; s < XC; ++s)
          if (s == qs) {
#pragma unroll
            for (int a = 0; a < RA; ++a) {
              const int i = lane + 64 * a;
              if (i > k && i < n) publish(true, i, x[s][a]);
            }
          }
      }
    } else {
      // the wave's four columns of threads summed: row lane + 64 a
#pragma unroll
      for (int a = 0; a < RA; ++a)
        spk[wave * NR + lane + 64 * a] =
            swap16_add(swap32_add(y[4 * a], y[4 * a + 2]), swap32_add(y[4 * a + 1], y[4 * a + 3]));
      if (tid >> 4 == (q & 15)) {
#pragma unroll
        for (int s = 0; s < XC; ++s)
          if (s == q >> 4) {
#pragma unroll
            for (int a = 0; a < XR; ++a) sck[ri + rd * a] = x[s][a];
          }
      }
    }
    if constexpr (MULTI) {
      constexpr int U = 2 * NR / TNT;
      const int L = n - k - 1;
      unsigned long long b[U];
#pragma unroll
      for (int u = 0; u < U; ++u) b[u] = TRI_MARK;
      for (int spin = 0; !dead; ++spin) {
        if (spin >= polls || (spin % TRI_LOOK == TRI_LOOK - 1 &&
                              __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          *gave = 1;
          atomicExch(status, 2);
          break;
        }
        bool more = false;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int e = tid + TNT * u;
          if (e < 2 * L && b[u] == TRI_MARK)
            b[u] = __hip_atomic_load(exk + (e < L ? k + 1 + e : n + k + 1 + (e - L)), __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) more = more || (tid + TNT * u < 2 * L && b[u] == TRI_MARK);
        if (!more) break;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = tid + TNT * u;
        if (e < 2 * L) (e < L ? spk[k + 1 + e] : sck[k + 1 + (e - L)]) = __longlong_as_double((long long)b[u]);
      }
    }
    lds_barrier();
    if constexpr (MULTI) dead = *gave != 0;
    // results of step k, stored here so that the trip through memory passes
    // behind the arithmetic and not before the next values are waited for
    if (MULTI ? gw == (qw ? qw - 1 : NWV - 1) : wave == (k & (TNW - 1))) {
#pragma unroll
      for (int a = 0; a < RA; ++a) {
        const int i = lane + 64 * a;
        if (i < n) V[size_t(k) * n + i] = v[a];
      }
      if (lane == 0) {
        ev[k] = al;
        tv[k] = tau;
      }
    }
    // w of step k, column k + 1 brought up to date, the next reflector
    double sm = 0.0;
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const int i = lane + 64 * a;
      const bool in = i > k && i < n;
      if constexpr (MULTI) {
        wp[a] = in ? spk[i] : 0.0;
      } else {
        double ps = spk[i];
#pragma unroll
        for (int w = 1; w < TNW; ++w) ps += spk[w * NR + i];
        wp[a] = in && tau != 0.0 ? tau * ps : 0.0;
      }
      c[a] = in ? sck[i] : 0.0;
      sm += v[a] * wp[a];
    }
    const double K = 0.5 * tau * wave_total(sm);
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      wp[a] -= K * v[a];
      vp[a] = v[a];
      lp[lane + 64 * a] = make_double2(v[a], wp[a]);
    }
    double vq, wq, x0;
    if constexpr (MULTI) {
      vq = lv[q];
      wq = spk[q] - K * vq;
      const double vq1 = lv[q + 1], wq1 = spk[q + 1] - K * vq1;
      x0 = sck[q + 1] - (vq1 * wq + wq1 * vq);
    } else {
      vq = pick(v, q);
      wq = pick(wp, q);
    }
#pragma unroll
    for (int a = 0; a < RA; ++a) c[a] -= v[a] * wq + wp[a] * vq;
    if constexpr (!MULTI) x0 = pick(c, q + 1);
    if (gw == 0 && lane == 0) dv[q] = sck[q] - (vq * wq + wq * vq);
    if (MULTI && ++qw == NWV) {
      qw = 0;
      ++qs;
    }
    if (q + 2 < n) {
      reflect(q, x0);
    } else if (gw == 0 && lane == 0) {
      ev[q] = x0;
    }
  }
  // the last diagonal element, with the pending update, from its owner
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const double2 pl = lp[n - 1];
#pragma unroll
  for (int s = 0; s < XC; ++s)
#pragma unroll
    for (int a = 0; a < XR; ++a)
      if (ci + cd * s == n - 1 && ri + rd * a == n - 1) {
        dv[n - 1] = x[s][a] - (pl.x * pl.y + pl.y * pl.x);
        ev[n - 1] = 0.0;
      }
}

// ---- Q times a matrix ---------------------------------------------------------
// X <- H_0 H_1 ... H_{n-3} X, one wave per QCB columns held in registers
// (lanes over rows): the columns are independent, so a wave applies all
// reflectors, last first, without meeting another one; the reflectors
// stream from the L2, QPF of them under way (with one the trip to the L2
// bounds the step: 78 us at n = 234, 68 with four or eight).  Bound by the
// latency of a reflector, 0.3 us: a dot product, its sum over the lanes and an
// update.  RA = ceil(n / 64) exactly (with the next power of two and four
// under way n = 300 took 177 us, now 101).
constexpr int QCB = 4;

template <int RA, int QPF>
__device__ __forceinline__ void back_run(const BackTask &tk, int c0, const double *__restrict__ W,
                                         const double *__restrict__ S, double *__restrict__ O,
                                         const int *__restrict__ rank) {
  const int n = tk.n, lane = threadIdx.x & 63;
  const double *__restrict__ V = W + tk.v_off;
  const double *__restrict__ tau = W + tk.d_off + 2 * size_t(n);
  double z[QCB][RA];
#pragma unroll
  for (int u = 0; u < QCB; ++u) {
    const int c = c0 + u;
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const int i = lane + 64 * a;
      z[u][a] = (c < n && i < n) ? S[tk.s_off + size_t(c) * n + i] : 0.0;
    }
  }
  // the next QPF reflectors are on their way while one is applied
  double v[QPF][RA], t[QPF];
  auto fetch = [&](int h, int k) {
    // from clamped places, zeroed after: no branch around the loads
    const int kc = max(k, 0);
    const double tk2 = tau[kc];
    t[h] = k >= 0 ? tk2 : 0.0;
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const int i = lane + 64 * a;
      const double x = V[size_t(kc) * n + min(i, n - 1)];
      v[h][a] = i < n ? x : 0.0;
    }
  };
#pragma unroll
  for (int h = 0; h < QPF; ++h) fetch(h, n - 3 - h);
  for (int k0 = n - 3; k0 >= 0; k0 -= QPF) {
#pragma unroll
    for (int h = 0; h < QPF; ++h) {  // past the first reflector: tau = 0
      double y[QCB];
#pragma unroll
      for (int u = 0; u < QCB; ++u) {
        y[u] = 0.0;
#pragma unroll
        for (int a = 0; a < RA; ++a) y[u] += v[h][a] * z[u][a];
      }
      const double s = t[h] * wave_totals<QCB>(y);
#pragma unroll
      for (int u = 0; u < QCB; ++u) {
        const double f = read_lane(s, u * (64 / QCB));
#pragma unroll
        for (int a = 0; a < RA; ++a) z[u][a] -= f * v[h][a];
      }
      fetch(h, k0 - h - QPF);
    }
  }
#pragma unroll
  for (int u = 0; u < QCB; ++u) {
    const int c = c0 + u;
    if (c >= n) continue;
    const size_t oc = size_t(rank[tk.r_off + c]);
#pragma unroll
    for (int a = 0; a < RA; ++a) {
      const int i = lane + 64 * a;
      if (i < n) O[tk.o_off + oc * n + i] = z[u][a];
    }
  }
}

}  // namespace
}  // namespace itx
