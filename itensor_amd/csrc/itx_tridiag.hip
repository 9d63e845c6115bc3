// Householder tridiagonal form of symmetric matrices, and products with its
// orthogonal factor: the dense O(n^3) parts of the symmetric eigensolver.
#include <algorithm>
#include <cstdlib>

#include "itx_tri.h"

namespace itx {
namespace {

// blocks[b] = (task, workgroup of the task)
__global__ __launch_bounds__(TNT) void k_tridiag(const TriTask *__restrict__ tasks, const int2 *__restrict__ blocks,
                                                 const double *__restrict__ A, double *__restrict__ W,
                                                 int *__restrict__ status, int polls) {
  __shared__ __align__(16) double lds[tri_lds<8, true>()];
  __shared__ int gave;  // a wave of this workgroup has given up a wait
  static_assert(tri_lds<8, true>() >= tri_lds<2, false>() && tri_lds<8, true>() >= tri_lds<4, true>(), "LDS of a class");
  const int2 b = blocks[blockIdx.x];
  const TriTask tk = tasks[b.x];
  int *st = status + b.x;
  if (threadIdx.x == 0) gave = 0;
  __syncthreads();
  if (tk.n <= 64)
    tri_run<1, false>(tk, 0, A, W, st, lds);
  else if (tk.n <= 128)
    tri_run<2, false>(tk, 0, A, W, st, lds);
  else if (tk.n <= 256)
    tri_run<4, true>(tk, b.y, A, W, st, lds, polls, &gave);
  else
    tri_run<8, true>(tk, b.y, A, W, st, lds, polls, &gave);
}

__global__ void k_mark(double *x, size_t n) {
  for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += size_t(gridDim.x) * blockDim.x)
    reinterpret_cast<unsigned long long *>(x)[i] = TRI_MARK;
}

// blocks[b] = (task, first of the block's 4 QCB columns)
__global__ __launch_bounds__(256) void k_back(const BackTask *__restrict__ tasks, const int2 *__restrict__ blocks,
                                              const double *__restrict__ W, const double *__restrict__ S,
                                              double *__restrict__ O, const int *__restrict__ rank,
                                              const int *__restrict__ status) {
  const int2 b = blocks[blockIdx.x];
  const BackTask tk = tasks[b.x];
  const int c0 = b.y + QCB * (threadIdx.x >> 6);
  if (c0 >= tk.n || status[b.x] != 0) return;  // no barrier below
  switch ((tk.n + 63) / 64) {
    case 1: return back_run<1, 8>(tk, c0, W, S, O, rank);
    case 2: return back_run<2, 8>(tk, c0, W, S, O, rank);
    case 3: return back_run<3, 8>(tk, c0, W, S, O, rank);
    case 4: return back_run<4, 8>(tk, c0, W, S, O, rank);
    case 5: return back_run<5, 8>(tk, c0, W, S, O, rank);
    case 6: return back_run<6, 8>(tk, c0, W, S, O, rank);
    case 7: return back_run<7, 8>(tk, c0, W, S, O, rank);
    default: return back_run<8, 8>(tk, c0, W, S, O, rank);
  }
}

}  // namespace

static int tri_wgs(int n) { return n <= 128 ? 1 : (n + TNW * TXC - 1) / (TNW * TXC); }

size_t tri_exchange(int n) { return n <= 128 ? 0 : size_t(n - 2) * 2 * size_t(n); }

TriWait tri_wait() {
  TriWait w;
  if (const char *v = std::getenv("ITX_EIG_WAIT")) {
    char *end = nullptr;
    w.polls = int(std::min(std::max(std::strtol(v, &end, 10), 0l), long(w.polls)));
    if (*end == ',') w.absent = std::atoi(end + 1) != 0;
  }
  return w;
}

void tri_blocks(std::vector<TriTask> &tasks, int ntasks, int cus, bool absent, std::vector<int2> &blocks,
                std::vector<size_t> &ends) {
  // Workgroups that meet come first, in launches of at most one workgroup
  // per CU, so that all of a launch are resident together.
  if (ntasks == 0) return;
  std::vector<int> order(static_cast<size_t>(ntasks));
  for (int i = 0; i < ntasks; ++i) {
    order[size_t(i)] = i;
    tasks[size_t(i)].wgs = tri_wgs(tasks[size_t(i)].n);
  }
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return tasks[size_t(x)].n > tasks[size_t(y)].n; });
  int meet = 0;
  for (int i : order) {
    const int g = tasks[size_t(i)].wgs;
    if (g > 1 && meet > 0 && meet + g > cus) {
      ends.push_back(blocks.size());
      meet = 0;
    }
    if (g > 1) meet += g;
    for (int b = 0; b < (absent && g > 1 ? g - 1 : g); ++b) blocks.push_back(make_int2(i, b));
  }
  ends.push_back(blocks.size());
}

void tri_launch(itx_ctx *ctx, const TriTask *tasks, const int2 *blocks, const std::vector<size_t> &ends,
                const double *A, double *W, int64_t x_off, size_t nx, int polls, int *status) {
  if (nx)
    hipLaunchKernelGGL(k_mark, dim3(unsigned(std::min<size_t>((nx + 255) / 256, size_t(ctx->num_cus) * 8))), dim3(256),
                       0, ctx->stream, W + x_off, nx);
  size_t start = 0;
  for (size_t e : ends) {
    if (e > start)
      hipLaunchKernelGGL(k_tridiag, dim3(unsigned(e - start)), dim3(TNT), 0, ctx->stream, tasks, blocks + start, A, W,
                         status, polls);
    start = e;
  }
}

void back_blocks(const std::vector<BackTask> &tasks, int ntasks, std::vector<int2> &blocks) {
  std::vector<int> order(static_cast<size_t>(ntasks));
  for (int i = 0; i < ntasks; ++i) order[size_t(i)] = i;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return tasks[size_t(x)].n > tasks[size_t(y)].n; });
  for (int i : order)
    for (int c = 0; c < tasks[size_t(i)].n; c += 4 * QCB) blocks.push_back(make_int2(i, c));
}

void back_launch(itx_ctx *ctx, const BackTask *tasks, const int2 *blocks, size_t nblocks, const double *W,
                 const double *S, double *O, const int *rank, const int *status) {
  if (nblocks)
    hipLaunchKernelGGL(k_back, dim3(unsigned(nblocks)), dim3(256), 0, ctx->stream, tasks, blocks, W, S, O, rank, status);
}

}  // namespace itx
