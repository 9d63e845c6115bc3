// Shared by the translation units of the symmetric eigensolver.
#pragma once

#include "itx_internal.h"

namespace itx {

// ---- wave reductions without LDS traffic ----------------------------------
// Lane exchanges by DPP inside a row of 16 lanes and by gfx950's permlane
// swaps across rows; every lane ends with the same bits.
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_ROR8 = 0x128;

template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, int(b), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double((long long)((unsigned long long)(unsigned)hi << 32 | (unsigned)lo));
}
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
// (a of the lower half, b of the lower half) + (a of the upper half, b of the upper half)
__device__ __forceinline__ double swap32_add(double a, double b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
  const u32x2 lo = __builtin_amdgcn_permlane32_swap(unsigned(x), unsigned(y), false, false);
  const u32x2 hi = __builtin_amdgcn_permlane32_swap(unsigned(x >> 32), unsigned(y >> 32), false, false);
  return __longlong_as_double((long long)((unsigned long long)hi.x << 32 | lo.x)) +
         __longlong_as_double((long long)((unsigned long long)hi.y << 32 | lo.y));
}
// the same within each half: rows (0, 1) and (2, 3)
__device__ __forceinline__ double swap16_add(double a, double b) {
  const unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
  const u32x2 lo = __builtin_amdgcn_permlane16_swap(unsigned(x), unsigned(y), false, false);
  const u32x2 hi = __builtin_amdgcn_permlane16_swap(unsigned(x >> 32), unsigned(y >> 32), false, false);
  return __longlong_as_double((long long)((unsigned long long)hi.x << 32 | lo.x)) +
         __longlong_as_double((long long)((unsigned long long)hi.y << 32 | lo.y));
}
// sum over the 64 lanes, in every lane (two FP64 MFMAs with ones instead of
// the six exchanges were measured slower: 330 more cycles a sum)
__device__ __forceinline__ double wave_total(double v) {
  v = swap32_add(v, v);
  v = swap16_add(v, v);
  v += dpp_move<DPP_ROR8>(v);
  v += dpp_move<DPP_HALF_MIRROR>(v);
  v += dpp_move<DPP_XOR2>(v);
  v += dpp_move<DPP_XOR1>(v);
  return v;
}
// Sums over the 64 lanes of NV values at once (NV = 4, 8, 16, 32): value t
// ends in the lanes t * 64 / NV ... (t + 1) * 64 / NV - 1.  Each exchange
// halves the number of values a lane carries, so NV sums take about NV
// additions instead of 6 NV.
template <int NV>
__device__ __forceinline__ double wave_totals(double (&y)[NV]) {
  static_assert(NV == 4 || NV == 8 || NV == 16 || NV == 32, "number of values");
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < NV / 2; ++q) y[q] = swap32_add(y[q], y[q + NV / 2]);
#pragma unroll
  for (int q = 0; q < NV / 4; ++q) y[q] = swap16_add(y[q], y[q + NV / 4]);
  auto half = [&](int n, int bit, auto mv) {  // n values left -> n / 2, selected by a lane bit
#pragma unroll
    for (int q = 0; q < n / 2; ++q) {
      const bool up = (lane & bit) != 0;
      const double z = up ? y[q + n / 2] : y[q], o = up ? y[q] : y[q + n / 2];
      y[q] = z + mv(o);
    }
  };
  if constexpr (NV >= 8)
    half(NV / 4, 8, [](double o) { return dpp_move<DPP_ROR8>(o); });
  else
    y[0] += dpp_move<DPP_ROR8>(y[0]);
  if constexpr (NV >= 16)
    half(NV / 8, 4, [](double o) { return dpp_move<DPP_HALF_MIRROR>(o); });
  else
    y[0] += dpp_move<DPP_HALF_MIRROR>(y[0]);
  if constexpr (NV >= 32)
    half(NV / 16, 2, [](double o) { return dpp_move<DPP_XOR2>(o); });
  else
    y[0] += dpp_move<DPP_XOR2>(y[0]);
  return y[0] + dpp_move<DPP_XOR1>(y[0]);
}
__device__ __forceinline__ double read_lane(double v, int l) {  // l wave-uniform
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane(unsigned(b), l), hi = __builtin_amdgcn_readlane(unsigned(b >> 32), l);
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// ---- reciprocals and square roots ---------------------------------------------
// The hardware estimate (24 bits) refined by Newton's iteration, one step of
// third order or two of second (error about one unit in the last place, for
// arguments well inside the normal range): a third of the dependent
// instructions of the division they stand for.
__device__ __forceinline__ double fast_rcp(double x) {
  const double r = __builtin_amdgcn_rcp(x), e = fma(-x, r, 1.0);
  return fma(fma(e, e, e), r, r);
}
__device__ __forceinline__ double fast_rsqrt(double x) {
  double r = __builtin_amdgcn_rsq(x);
  r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
  return fma(0.5 * r, fma(-x * r, r, 1.0), r);
}
__device__ __forceinline__ double fast_sqrt(double x) {  // x = 0 gives 0
  double r = __builtin_amdgcn_rsq(x);
  r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
  const double s = x * r;
  return x > 0.0 ? fma(fma(-s, s, x), 0.5 * r, s) : 0.0;
}

// ---- Householder tridiagonal form (itx_tridiag.hip) -------------------------
// One symmetric matrix: A (column-major, both triangles) at a_off of the
// caller's array; the rest in the workspace: V (n x n, column k the
// reflector v_k, zero down to row k; columns 0 .. n-3), then d, e and tau
// (n each) at d_off, the exchange area at x_off (several workgroups only).
struct TriTask {
  int32_t n, wgs;
  int64_t a_off, v_off, d_off, x_off;
};
constexpr int TRI_MAX = 512;  // largest order
// exchange doubles of a matrix of order n
size_t tri_exchange(int n);
// How long a workgroup waits for the others of its matrix: 2^20 polls, about
// a second.  ITX_EIG_WAIT=polls[,1] shortens it for tests (0: every wait is
// given up at once; 1: the last workgroup of each matrix is not launched).
struct TriWait {
  int polls = 1 << 20;
  bool absent = false;
};
TriWait tri_wait();
// Sets the workgroup count of the first ntasks tasks and lists the
// workgroups (task, workgroup) in launch order; ends: the end of each launch
// in the list.
void tri_blocks(std::vector<TriTask> &tasks, int ntasks, int cus, bool absent, std::vector<int2> &blocks,
                std::vector<size_t> &ends);
// Reduces every task: T = Q^T A Q, Q = H_0 H_1 ... H_{n-3}, H_k = I - tau_k
// v_k v_k^T.  tasks, blocks: device copies; W: workspace, whose exchange
// area is the nx doubles at x_off; status: one int per task (zero before the
// call), set to 2 where the workgroups of a matrix did not meet.
void tri_launch(itx_ctx *ctx, const TriTask *tasks, const int2 *blocks, const std::vector<size_t> &ends,
                const double *A, double *W, int64_t x_off, size_t nx, int polls, int *status);
// O <- Q S for the n x n matrix of every task: column c of S (at s_off) goes
// to column rank[r_off + c] of O.  Tasks with a status are left out.
struct BackTask {
  int32_t n, pad;
  int64_t v_off, d_off, s_off, o_off, r_off;
};
void back_blocks(const std::vector<BackTask> &tasks, int ntasks, std::vector<int2> &blocks);
void back_launch(itx_ctx *ctx, const BackTask *tasks, const int2 *blocks, size_t nblocks, const double *W,
                 const double *S, double *O, const int *rank, const int *status);

// ---- divide and conquer (itx_dc.hip) -----------------------------------------
// One tridiagonal matrix: d, e at d_off of the workspace (as TriTask), four
// n x n matrices from q_off (the vectors, twice; the secular problems'
// differences and vectors), AUX_SIZE(n) doubles at x_off.  Eigenvalues go to
// w_off of w, and to r_off of the host's and of the rank array.
struct DcTask {
  int32_t n, p;  // p: 2^p leaves
  int64_t d_off, x_off, q_off, r_off, w_off;
};
constexpr int DC_MAX = 512;
__host__ __device__ constexpr size_t AUX_D(int n, int par) { return size_t(par) * n; }  // eigenvalues, by level parity
__host__ __device__ constexpr size_t AUX_DS(int n) { return 2 * size_t(n); }            // poles
__host__ __device__ constexpr size_t AUX_ZS(int n) { return 3 * size_t(n); }            // their z
__host__ __device__ constexpr size_t AUX_SEL(int n) { return 4 * size_t(n); }           // column of each (int)
__host__ __device__ constexpr size_t AUX_K(int n) { return 5 * size_t(n); }             // poles of a merge (int)
__host__ __device__ constexpr size_t AUX_SCALE(int n) { return 6 * size_t(n); }             // of d and e; infinite: unscaled, e ignored
__host__ __device__ constexpr size_t AUX_SIZE(int n) { return 6 * size_t(n) + 2; }
inline int dc_levels(int n) {
  int p = 0;
  while ((1 << p) < n) ++p;
  return p;
}
// where the eigenvectors end, relative to q_off
inline int64_t dc_vectors(int n) {
  const int p = dc_levels(n);
  return p > 6 && ((p - 6) & 1) ? int64_t(n) * n : 0;
}
// Where results go: ranks (device), eigenvalues and states for the host
// (coherent pinned memory), the states on the device, the counter of
// finished matrices (zero before the call) and the host's flag, set to seq
// by the last of `count` matrices.
struct DcOut {
  int *rank;
  double *hw;
  int *status, *hstatus;
  unsigned *done;
  unsigned long long *flag, seq;
  int count;
};
// The workgroups (task, node) of the 64-row subtrees of the first ntasks
// tasks (all above 64 rows), then of every level above.
struct DcLevel {
  int level;
  size_t first, count;
  int maxm;  // largest merge
};
void dc_blocks(const std::vector<DcTask> &tasks, int ntasks, std::vector<int2> &blocks, std::vector<DcLevel> &levels);
// Eigenvalues and vectors of the tridiagonal matrices of the first ntasks tasks.
void dc_launch(itx_ctx *ctx, const DcTask *tasks, int ntasks, const int2 *blocks, const std::vector<DcLevel> &levels,
               double *W, double *w, const DcOut &out);
// Whole decomposition of the tasks first .. first + count - 1, at most 64 rows each.
void syev_small_launch(itx_ctx *ctx, const TriTask *tri, const DcTask *tasks, const BackTask *back, int first, int count,
                       double *A, double *W, double *w, const DcOut &out);

}  // namespace itx
