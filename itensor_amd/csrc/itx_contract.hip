// Contraction engine of libitx: dense and block-sparse (QN) tensor
// contractions as one persistent MFMA GEMM kernel with the index
// permutations folded into offset-table driven tile loads and stores.
//
// Reference behaviour replaced:
//   contract() / CProps (tensor/contract.cc:137-866) reduces a binary
//   contraction to permute(A), permute(B) -> dgemm -> permute(C).  Here the
//   permutations never touch memory: the plan records, for every logical
//   row m, column n and contracted position k of the GEMM, the element
//   offset inside each operand (tables aM,aK,bK,bN,cM,cN), so the kernel
//   gathers tiles straight from the original layouts.
//   doTask(Contract,QDense,QDense) (itdata/qdense.cc:671-743) runs one
//   contract() per (A block, B block) pair; here all pairs of one
//   contraction are tasks of a single launch, grouped by C block so that
//   all pairs feeding one C tile are summed in registers (the reference's
//   OpenMP path groups by output block for the same reason,
//   itdata/qutil.h:271-349).
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdio>
#include <fstream>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <numeric>
#include <queue>
#include <sstream>
#include <type_traits>
#include <utility>

#include <unordered_map>
#include "itx_internal.h"

namespace itx {
namespace {

constexpr int BK = 16;   // K depth of one LDS stage (default)

template <typename T>
struct MF;
template <>
struct MF<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // swizzle of LDS columns per K row (keeps 8-byte accesses conflict free)
  static __device__ __forceinline__ int sw(int k) { return (k >> 1) & 7; }
  // output row of accumulator element r held by `lane` (measured on gfx950:
  // the f64 16x16x4 result interleaves rows, row = lane/16 + 4r)
  static __device__ __forceinline__ int orow(int lane, int r) { return (lane >> 4) + 4 * r; }
  template <int BMX>
  static constexpr int pad() { return 16; }
};
template <>
struct MF<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int sw(int k) { return (k >> 2) & 3; }
  // f32 16x16x4 result: blocked rows, row = 4*(lane/16) + r
  static __device__ __forceinline__ int orow(int lane, int r) { return 4 * (lane >> 4) + r; }
  template <int BMX>
  static constexpr int pad() { return BMX == 32 ? 48 : 16; }
};

// Loader of one operand tile (rows x BK) into LDS laid out [k][row].
// KC: the operand is contiguous along k (lanes walk k), else along rows.
// The k-offset table entries of a stage are fetched one stage ahead
// (fetch_k) so that the data loads of the next stage never wait on a table
// read, and every load is issued unconditionally from a clamped address
// (out-of-range elements read element 0 of the block and are zeroed), which
// keeps the load stream free of exec-mask branches.
// Offsets stay 64-bit: 32-bit offsets measured 1.6x slower on gfx950.
// With V = 2 (k-contiguous operands whose k runs come in aligned pairs,
// checked when the plan is built) a lane loads two consecutive k of one
// row as one 16-byte load and fetches one table entry per pair.
template <typename T, int BR, bool KC, int NTH, int BK = 16, int V = 1>
struct TileLoader {
  static constexpr int PER = BR * BK / NTH;  // elements per thread
  static_assert(PER >= 1, "tile too small for the thread count");
  static_assert(V == 1 || (KC && PER % V == 0 && BK % V == 0), "vector loads need a k-contiguous operand");
  static constexpr int NV = PER / V;         // loads per thread
  static constexpr int LK = BK / V;          // lanes along k (KC)
  static constexpr int LD = BR + MF<T>::template pad<BR>();
  static constexpr int NK = KC ? 1 : PER;  // k offsets per thread and stage
  double r[PER];
  bool rok[NV];  // element in range (applied at store, after the MFMAs)
  int64_t roff[KC ? NV : 1];
  bool rv[KC ? NV : 1];
  int64_t ko[NK];
  bool kv[NK];
  int lr, lk;  // thread's base row / base k

  __device__ __forceinline__ void init(int tid, int row0, int R, const int64_t *__restrict__ tabR) {
    if constexpr (KC) {
      lk = (tid % LK) * V;
      lr = tid / LK;
#pragma unroll
      for (int p = 0; p < NV; ++p) {
        int row = row0 + lr + (NTH / LK) * p;
        rv[p] = row < R;
        roff[p] = tabR[rv[p] ? row : 0];
      }
    } else {
      lr = tid % BR;
      lk = tid / BR;
      int row = row0 + lr;
      rv[0] = row < R;
      roff[0] = tabR[rv[0] ? row : 0];
    }
  }
  // table reads for the stage starting at k0
  __device__ __forceinline__ void fetch_k(int k0, int K, const int64_t *__restrict__ tabK) {
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      const int k = k0 + lk + (KC ? 0 : (NTH / BR) * q);
      kv[q] = k < K;
      ko[q] = tabK[kv[q] ? k : 0];
    }
  }
  // data loads of the stage whose offsets fetch_k last read
  __device__ __forceinline__ void load(const double *__restrict__ base) {
#pragma unroll
    for (int p = 0; p < NV; ++p) {
      const bool ok = KC ? (kv[0] && rv[p]) : (kv[p] && rv[0]);
      const int64_t off = (KC ? roff[p] + ko[0] : roff[0] + ko[p]);
      if constexpr (V == 2) {
        const double2 v = *reinterpret_cast<const double2 *>(base + (ok ? off : 0));
        r[2 * p] = v.x;
        r[2 * p + 1] = v.y;
      } else {
        r[p] = base[ok ? off : 0];
      }
      rok[p] = ok;
    }
  }
  __device__ __forceinline__ void store(T *__restrict__ s) const {
    if constexpr (KC) {
#pragma unroll
      for (int p = 0; p < NV; ++p) {
        int row = lr + (NTH / LK) * p;
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const int k = lk + e;
          s[k * LD + (row ^ MF<T>::sw(k))] = rok[p] ? T(r[V * p + e]) : T(0);
        }
      }
    } else {
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        int k = lk + (NTH / BR) * p;
        s[k * LD + (lr ^ MF<T>::sw(k))] = rok[p] ? T(r[p]) : T(0);
      }
    }
  }
};

// One workgroup = GM x GN waves computing a BM x BN tile of C; each wave
// owns a (BM/GM) x (BN/GN) sub-tile of 16x16 MFMA fragments.
template <typename T, int BM, int BN, int GM, int GN, bool AKC, bool BKC, int BK, int V>
__global__ __launch_bounds__(64 * GM * GN) void k_gemm(const double *__restrict__ A, const double *__restrict__ B,
                                                       double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                       const WorkUnit *__restrict__ units, int nunits,
                                                       const int64_t *__restrict__ tab, double alpha, double beta) {
  constexpr int NTH = 64 * GM * GN;
  using v4 = typename MF<T>::v4;
  using LA = TileLoader<T, BM, AKC, NTH, BK, V>;
  using LB = TileLoader<T, BN, BKC, NTH, BK, V>;
  constexpr int WM = BM / GM, WN = BN / GN, FM = WM / 16, FN = WN / 16;
  static_assert(FM >= 1 && FN >= 1, "wave tile below one MFMA fragment");
  __shared__ T As[2][BK * LA::LD];
  __shared__ T Bs[2][BK * LB::LD];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % GM, wn = wave / GM;

  // the planner has dealt the list to the XCDs (blocks b with equal b % 8)
  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    v4 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = v4{0, 0, 0, 0};

    for (int t = wu.tbeg; t < wu.tend; ++t) {
      const GemmTask tk = tasks[t];
      if (tk.K <= 0) continue;
      LA la;
      LB lb;
      la.init(tid, wu.m0, tk.M, tab + tk.tAM);
      lb.init(tid, wu.n0, tk.N, tab + tk.tBN);
      const double *Ab = A + tk.a_off;
      const double *Bb = B + tk.b_off;
      const int64_t *tAK = tab + tk.tAK;
      const int64_t *tBK = tab + tk.tBK;
      la.fetch_k(0, tk.K, tAK);
      lb.fetch_k(0, tk.K, tBK);
      la.load(Ab);
      lb.load(Bb);
      la.fetch_k(BK, tk.K, tAK);
      lb.fetch_k(BK, tk.K, tBK);
      la.store(As[0]);
      lb.store(Bs[0]);
      __syncthreads();
      int cur = 0;
      for (int k0 = 0; k0 < tk.K; k0 += BK) {
        const bool nxt = k0 + BK < tk.K;
        if (nxt) {
          la.load(Ab);  // stage k0+BK (offsets fetched one stage earlier)
          lb.load(Bb);
          la.fetch_k(k0 + 2 * BK, tk.K, tAK);
          lb.fetch_k(k0 + 2 * BK, tk.K, tBK);
        }
        const T *as = As[cur];
        const T *bs = Bs[cur];
#pragma unroll
        for (int kq = 0; kq < BK / 4; ++kq) {
          const int kr = kq * 4 + (lane >> 4);
          T af[FM], bf[FN];
#pragma unroll
          for (int j = 0; j < FM; ++j) {
            int m = wm * WM + j * 16 + (lane & 15);
            af[j] = as[kr * LA::LD + (m ^ MF<T>::sw(kr))];
          }
#pragma unroll
          for (int i = 0; i < FN; ++i) {
            int n = wn * WN + i * 16 + (lane & 15);
            bf[i] = bs[kr * LB::LD + (n ^ MF<T>::sw(kr))];
          }
          // D^T tile: MFMA rows run over n, columns over m, so that the
          // 16 lanes of a row hold 16 consecutive m (coalesced C stores).
#pragma unroll
          for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j) acc[i][j] = MF<T>::mma(bf[i], af[j], acc[i][j]);
        }
        if (nxt) {
          la.store(As[cur ^ 1]);
          lb.store(Bs[cur ^ 1]);
        }
        __syncthreads();
        cur ^= 1;
      }
    }

    // epilogue: C = alpha*acc + beta*C through the C offset tables
    const GemmTask t0 = tasks[wu.tbeg];
    const int64_t *tCM = tab + t0.tCM;
    const int64_t *tCN = tab + t0.tCN;
    double *Cb = C + t0.c_off;
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = wu.m0 + wm * WM + j * 16 + (lane & 15);
      if (m >= t0.M) continue;
      const int64_t cm = tCM[m];
#pragma unroll
      for (int i = 0; i < FN; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = wu.n0 + wn * WN + i * 16 + MF<T>::orow(lane, r);
          if (n < t0.N) {
            const int64_t ad = cm + tCN[n];
            double v = alpha * double(acc[i][j][r]);
            if (beta != 0.0) v += beta * Cb[ad];
            Cb[ad] = v;
          }
        }
      }
    }
  }
}

// ---- register-pipelined tiles ---------------------------------------------
// FP64: k_pipe below.  FP32 (k_dgemm): 128 x 128 C tile, four waves of 64 x
// 64 (4 x 4 fragments of the f32 16x16x4 MFMA), 16-deep k stages, for
// operands contiguous along k in aligned pairs (the plan's vector-load
// condition).  A thread loads 16-byte k pairs and rounds them to FP32 at the
// LDS store; an LDS row holds the 16 k of a stage contiguously (pitch 18
// doubles, 20 floats: the 16 rows that a quarter-wave reads land on distinct
// 16-byte bank groups), and a lane reads the 4 consecutive k of its fragment
// row with 16-byte reads.  MFMA s (0..3) of a stage takes k = 4q + s from the
// lanes of quarter q, so every k of the stage enters once.
// Pipeline (one barrier per stage): while the MFMAs of stage n run from
// registers, the operands of stage n+1 are read from LDS, stage n+2 is
// stored to LDS from the load registers, and the global loads of stage n+4
// are issued into those registers (two register sets: loads have two
// stages to arrive).
constexpr int DG_BK = 16, DG_NT = 256;
template <typename T>
struct DgCfg;
template <>
struct DgCfg<double> {
  static constexpr int P = 18;  // LDS row pitch (elements)
};
template <>
struct DgCfg<float> {
  static constexpr int P = 20;
  static constexpr int RD = 8;  // LDS reads per stage and lane
};

struct DgRegs {  // one stage of one operand in flight: four 16-byte pairs
  double g[8];
  bool ok[4];
};

struct DgLoader {  // one operand: 128 rows x 16 k per stage, four 16-byte loads per thread
  int64_t roff[4];
  bool rv[4];
  int64_t ko[2];  // k offsets of the next two stages to load (slot = stage & 1)
  bool kv[2];
  int lr, lc;  // base row (32 rows apart per load), k pair
  __device__ __forceinline__ void init(int tid, int row0, int R, const int64_t *__restrict__ tabR) {
    lc = tid & 7;
    lr = tid >> 3;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int row = row0 + lr + 32 * p;
      rv[p] = row < R;
      roff[p] = tabR[rv[p] ? row : 0];
    }
  }
  __device__ __forceinline__ void fetch_k(int k0, int K, const int64_t *__restrict__ tabK, int slot) {
    const int k = k0 + 2 * lc;  // K is even: the pair is in range with its first k
    kv[slot] = k < K;
    ko[slot] = tabK[kv[slot] ? k : 0];
  }
  __device__ __forceinline__ void load(const double *__restrict__ base, DgRegs &r, int slot) const {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      r.ok[p] = kv[slot] && rv[p];
      const double2 v = *reinterpret_cast<const double2 *>(base + (r.ok[p] ? roff[p] + ko[slot] : 0));
      r.g[2 * p] = v.x;
      r.g[2 * p + 1] = v.y;
    }
  }
  __device__ __forceinline__ void store(float *__restrict__ s, const DgRegs &r) const {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      float2 v;
      v.x = r.ok[p] ? float(r.g[2 * p]) : 0.0f;
      v.y = r.ok[p] ? float(r.g[2 * p + 1]) : 0.0f;
      *reinterpret_cast<float2 *>(s + (lr + 32 * p) * DgCfg<float>::P + 2 * lc) = v;
    }
  }
};

template <typename T>
struct DgFrag;
template <>
struct DgFrag<float> {  // a lane's operands of one stage: 4 fragments x 4 k, for A and for B
  float4 a[4], b[4];
};

__device__ __forceinline__ void dg_read(DgFrag<float> &f, const float *__restrict__ as, const float *__restrict__ bs,
                                        int wm, int wn, int lane) {
  const int r = lane & 15, q = lane >> 4;
  constexpr int P = DgCfg<float>::P;
#pragma unroll
  for (int j = 0; j < 4; ++j) f.a[j] = *reinterpret_cast<const float4 *>(as + (wm * 64 + j * 16 + r) * P + 4 * q);
#pragma unroll
  for (int i = 0; i < 4; ++i) f.b[i] = *reinterpret_cast<const float4 *>(bs + (wn * 64 + i * 16 + r) * P + 4 * q);
}

__device__ __forceinline__ double dg_k(const double2 (&x)[2], int s) {
  return s == 0 ? x[0].x : s == 1 ? x[0].y : s == 2 ? x[1].x : x[1].y;
}
__device__ __forceinline__ float dg_k(const float4 &x, int s) {
  return s == 0 ? x.x : s == 1 ? x.y : s == 2 ? x.z : x.w;
}

// the 16 MFMAs of k slot s (k = 4q + s in quarter q)
template <typename T>
__device__ __forceinline__ void dg_mfma(typename MF<T>::v4 (&acc)[4][4], const DgFrag<T> &f, int s) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = MF<T>::mma(dg_k(f.b[i], s), dg_k(f.a[j], s), acc[i][j]);
}

template <typename T>
__global__ __launch_bounds__(DG_NT) void k_dgemm(const double *__restrict__ A, const double *__restrict__ B,
                                                 double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                 const WorkUnit *__restrict__ units, int nunits,
                                                 const int64_t *__restrict__ tab, double alpha, double beta) {
  using v4 = typename MF<T>::v4;
  constexpr int P = DgCfg<T>::P, RD = DgCfg<T>::RD;
  __shared__ __align__(16) T As[2][128 * P];
  __shared__ __align__(16) T Bs[2][128 * P];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;

  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    v4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = v4{0, 0, 0, 0};

    for (int t = wu.tbeg; t < wu.tend; ++t) {
      const GemmTask tk = tasks[t];
      if (tk.K <= 0) continue;
      DgLoader la, lb;
      la.init(tid, wu.m0, tk.M, tab + tk.tAM);
      lb.init(tid, wu.n0, tk.N, tab + tk.tBN);
      const double *Ab = A + tk.a_off;
      const double *Bb = B + tk.b_off;
      const int64_t *tAK = tab + tk.tAK;
      const int64_t *tBK = tab + tk.tBK;
      const int S = (tk.K + DG_BK - 1) / DG_BK;
      DgRegs ra0, rb0, ra1, rb1;  // load register sets
// load stage st (its k offsets fetched two loads ago, slot st & 1) and
// fetch the k offsets of stage st + 2 into the same slot: a table read then
// never waits behind the data loads just issued
#define ITX_DG_LOAD(st, ra, rb, slot)                      \
  {                                                        \
    la.load(Ab, ra, slot);                                 \
    lb.load(Bb, rb, slot);                                 \
    la.fetch_k(((st) + 2) * DG_BK, tk.K, tAK, slot);       \
    lb.fetch_k(((st) + 2) * DG_BK, tk.K, tBK, slot);       \
  }
      // prologue: stages 0 and 1 into LDS, stage 0 into registers, stage 2
      // in set 1 and stage 3 in set 0
      la.fetch_k(0, tk.K, tAK, 0);
      lb.fetch_k(0, tk.K, tBK, 0);
      la.fetch_k(DG_BK, tk.K, tAK, 1);
      lb.fetch_k(DG_BK, tk.K, tBK, 1);
      ITX_DG_LOAD(0, ra0, rb0, 0)
      __syncthreads();  // the previous task's LDS reads are done
      la.store(As[0], ra0);
      lb.store(Bs[0], rb0);
      if (S > 1) ITX_DG_LOAD(1, ra0, rb0, 1)
      if (S > 2) ITX_DG_LOAD(2, ra1, rb1, 0)
      __syncthreads();
      DgFrag<T> f0, f1;
      dg_read(f0, As[0], Bs[0], wm, wn, lane);
      if (S > 1) {
        la.store(As[1], ra0);
        lb.store(Bs[1], rb0);
      }
      if (S > 3) ITX_DG_LOAD(3, ra0, rb0, 1)
      __syncthreads();
      // stage n: its MFMAs from registers; stage n+1 read from LDS[(n+1)&1]
      // at the start; after the first 16 MFMAs, stage n+2 stored from its
      // register set into LDS[n&1] (read into registers one stage ago) and
      // the loads of stage n+4 issued into that set.  The scheduling
      // barriers keep the store and the loads inside the MFMA stream and the
      // workgroup barrier behind the last MFMA (the stores have long
      // completed when the waves meet there).
#define ITX_DG_STEP(n, cur, nxt, ra, rb, slot)                                        \
  {                                                                               \
    if ((n) + 1 < S) dg_read(nxt, As[((n) + 1) & 1], Bs[((n) + 1) & 1], wm, wn, lane); \
    dg_mfma(acc, cur, 0);                                                         \
    __builtin_amdgcn_sched_barrier(0);                                            \
    if ((n) + 2 < S) {                                                            \
      la.store(As[(n) & 1], ra);                                                  \
      lb.store(Bs[(n) & 1], rb);                                                  \
    }                                                                             \
    if ((n) + 4 < S) ITX_DG_LOAD((n) + 4, ra, rb, slot)                           \
    __builtin_amdgcn_sched_barrier(0);                                            \
    dg_mfma(acc, cur, 1);                                                         \
    dg_mfma(acc, cur, 2);                                                         \
    dg_mfma(acc, cur, 3);                                                         \
    __builtin_amdgcn_sched_barrier(0);                                            \
    __syncthreads();                                                              \
  }
      // Steady state (stages n with n+4 < S): the same work without
      // conditions, in one scheduling region, with the LDS reads, the LDS
      // stores (and their selects) and the global loads (and their address
      // arithmetic) placed between consecutive MFMAs, so that the MFMA pipe
      // never waits on the wave's other instructions.
#define ITX_DG_BODY(n, cur, nxt, ra, rb, id)                                      \
  {                                                                               \
    dg_read(nxt, As[((n) + 1) & 1], Bs[((n) + 1) & 1], wm, wn, lane);            \
    dg_mfma(acc, cur, 0);                                                         \
    for (int g_ = 0; g_ < RD; ++g_) {                                             \
      __builtin_amdgcn_sched_group_barrier(0x008, 16 / RD, id);                   \
      __builtin_amdgcn_sched_group_barrier(0x100, 1, id);                         \
    }                                                                             \
    __builtin_amdgcn_sched_barrier(0);                                            \
    la.store(As[(n) & 1], ra);                                                    \
    lb.store(Bs[(n) & 1], rb);                                                    \
    dg_mfma(acc, cur, 1);                                                         \
    for (int g_ = 0; g_ < 8; ++g_) {                                              \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, id);                         \
      __builtin_amdgcn_sched_group_barrier(0x006, 4, id);                         \
      __builtin_amdgcn_sched_group_barrier(0x200, 1, id);                         \
    }                                                                             \
    __builtin_amdgcn_sched_group_barrier(0x008, 8, id);                           \
    __builtin_amdgcn_sched_barrier(0);                                            \
    ITX_DG_LOAD((n) + 4, ra, rb, id)                                              \
    dg_mfma(acc, cur, 2);                                                         \
    for (int g_ = 0; g_ < 12; ++g_) {                                             \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, id);                         \
      __builtin_amdgcn_sched_group_barrier(0x006, 6, id);                         \
      __builtin_amdgcn_sched_group_barrier(0x020, 1, id);                         \
    }                                                                             \
    __builtin_amdgcn_sched_group_barrier(0x008, 4, id);                           \
    __builtin_amdgcn_sched_barrier(0);                                            \
    dg_mfma(acc, cur, 3);                                                         \
    __builtin_amdgcn_sched_barrier(0);                                            \
    __syncthreads();                                                              \
  }
      int n = 0;
      for (; n + 5 < S; n += 2) {
        ITX_DG_BODY(n, f0, f1, ra1, rb1, 0)
        ITX_DG_BODY(n + 1, f1, f0, ra0, rb0, 1)
      }
      for (; n + 1 < S; n += 2) {
        ITX_DG_STEP(n, f0, f1, ra1, rb1, 0)
        ITX_DG_STEP(n + 1, f1, f0, ra0, rb0, 1)
      }
      if (n < S) ITX_DG_STEP(n, f0, f1, ra1, rb1, 0)
#undef ITX_DG_BODY
#undef ITX_DG_STEP
#undef ITX_DG_LOAD
    }

    // epilogue: C = alpha*acc + beta*C through the C offset tables (the
    // table entries of all of the lane's rows and columns are read before
    // the first store, from clamped indices)
    const GemmTask t0 = tasks[wu.tbeg];
    const int64_t *tCM = tab + t0.tCM;
    const int64_t *tCN = tab + t0.tCN;
    double *Cb = C + t0.c_off;
    int64_t cm[4], cn[4][4];
    bool mv[4], nv[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = wu.m0 + wm * 64 + j * 16 + (lane & 15);
      mv[j] = m < t0.M;
      cm[j] = tCM[mv[j] ? m : 0];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = wu.n0 + wn * 64 + i * 16 + MF<T>::orow(lane, r);
        nv[i][r] = n < t0.N;
        cn[i][r] = tCN[nv[i][r] ? n : 0];
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (mv[j] && nv[i][r]) {
            const int64_t ad = cm[j] + cn[i][r];
            double v = alpha * double(acc[i][j][r]);
            if (beta != 0.0) v += beta * Cb[ad];
            Cb[ad] = v;
          }
        }
  }
}

// ---- FP64 tile, two workgroups per CU ------------------------------------
// The tile, LDS layout and k order of k_dgemm (results bit for bit equal),
// with the register budget of two waves per SIMD (128 accumulator + at most
// 128 other registers): the operands are read from LDS one k slot ahead
// (16 MFMAs) instead of one stage ahead, and one set of load registers
// holds the next stage.  Two resident workgroups per CU cover each other's
// barrier waits, epilogues and first loads.  One barrier per stage, before
// the last slot, which reads the next stage's first slot.
template <typename T>
struct DgSlot {  // a lane's operands of one k slot: 4 A and 4 B fragments
  T a[4], b[4];
};

template <typename T>
__device__ __forceinline__ void dg_read_slot(DgSlot<T> &f, const T *__restrict__ as, const T *__restrict__ bs,
                                             int wm, int wn, int lane, int s) {
  const int r = lane & 15, q = lane >> 4;
  constexpr int P = DgCfg<T>::P;
#pragma unroll
  for (int j = 0; j < 4; ++j) f.a[j] = as[(wm * 64 + j * 16 + r) * P + 4 * q + s];
#pragma unroll
  for (int i = 0; i < 4; ++i) f.b[i] = bs[(wn * 64 + i * 16 + r) * P + 4 * q + s];
}

template <typename T>
__device__ __forceinline__ void dg_mfma_slot(typename MF<T>::v4 (&acc)[4][4], const DgSlot<T> &f) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = MF<T>::mma(f.b[i], f.a[j], acc[i][j]);
}

template <typename T>
__global__ __launch_bounds__(DG_NT, 2) void k_dgemm2(const double *__restrict__ A, const double *__restrict__ B,
                                                     double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                     const WorkUnit *__restrict__ units, int nunits,
                                                     const int64_t *__restrict__ tab, double alpha, double beta) {
  using v4 = typename MF<T>::v4;
  constexpr int P = DgCfg<T>::P;
  __shared__ __align__(16) T As[2][128 * P];
  __shared__ __align__(16) T Bs[2][128 * P];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;


  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    v4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = v4{0, 0, 0, 0};

    for (int t = wu.tbeg; t < wu.tend; ++t) {
      const GemmTask tk = tasks[t];
      if (tk.K <= 0) continue;
      DgLoader la, lb;
      la.init(tid, wu.m0, tk.M, tab + tk.tAM);
      lb.init(tid, wu.n0, tk.N, tab + tk.tBN);
      const double *Ab = A + tk.a_off;
      const double *Bb = B + tk.b_off;
      const int64_t *tAK = tab + tk.tAK;
      const int64_t *tBK = tab + tk.tBK;
      const int K = tk.K, S = (K + DG_BK - 1) / DG_BK;
      DgRegs ra, rb;
// load stage st and fetch the k offsets of stage st + 1 (one slot: with two
// workgroups per CU the table read's wait behind the data loads is covered)
#define ITX_DG2_LOAD(st, sl)                                  \
  {                                                           \
    la.load(Ab, ra, 0);                                       \
    lb.load(Bb, rb, 0);                                       \
    la.fetch_k(((st) + 1) * DG_BK, K, tAK, 0);                \
    lb.fetch_k(((st) + 1) * DG_BK, K, tBK, 0);                \
  }
      la.fetch_k(0, K, tAK, 0);
      lb.fetch_k(0, K, tBK, 0);
      ITX_DG2_LOAD(0, 0)
      __syncthreads();  // the previous task's LDS reads are done
      la.store(As[0], ra);
      lb.store(Bs[0], rb);
      if (S > 1) ITX_DG2_LOAD(1, 1)
      __syncthreads();
      DgSlot<T> cur, nxt;
      dg_read_slot(cur, As[0], Bs[0], wm, wn, lane, 0);
      // stage n (buffer n & 1, load slot sl = n & 1): stage n+1 (in the load
      // registers) into the other buffer, whose stage n-1 reads ended before
      // the previous barrier; the loads of stage n+2; the four k slots, each
      // reading the next slot's operands
#define ITX_DG2_STAGE(n, sl)                                                      \
  {                                                                               \
    const T *as = As[sl], *bs = Bs[sl];                                           \
    if ((n) + 1 < S) {                                                            \
      la.store(As[(sl) ^ 1], ra);                                                 \
      lb.store(Bs[(sl) ^ 1], rb);                                                 \
    }                                                                             \
    if ((n) + 2 < S) ITX_DG2_LOAD((n) + 2, sl)                                    \
    dg_read_slot(nxt, as, bs, wm, wn, lane, 1);                                   \
    dg_mfma_slot(acc, cur);                                                       \
    dg_read_slot(cur, as, bs, wm, wn, lane, 2);                                   \
    dg_mfma_slot(acc, nxt);                                                       \
    dg_read_slot(nxt, as, bs, wm, wn, lane, 3);                                   \
    dg_mfma_slot(acc, cur);                                                       \
    __syncthreads(); /* stage n+1 stored by every wave; stage n's reads done */   \
    if ((n) + 1 < S) dg_read_slot(cur, As[(sl) ^ 1], Bs[(sl) ^ 1], wm, wn, lane, 0); \
    dg_mfma_slot(acc, nxt);                                                       \
  }
      int n = 0;
      for (; n + 1 < S; n += 2) {
        ITX_DG2_STAGE(n, 0)
        ITX_DG2_STAGE(n + 1, 1)
      }
      if (n < S) ITX_DG2_STAGE(n, 0)
#undef ITX_DG2_STAGE
#undef ITX_DG2_LOAD
    }

    const GemmTask t0 = tasks[wu.tbeg];
    const int64_t *tCM = tab + t0.tCM;
    const int64_t *tCN = tab + t0.tCN;
    double *Cb = C + t0.c_off;
    int64_t cm[4], cn[4][4];
    bool mv[4], nv[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = wu.m0 + wm * 64 + j * 16 + (lane & 15);
      mv[j] = m < t0.M;
      cm[j] = tCM[mv[j] ? m : 0];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = wu.n0 + wn * 64 + i * 16 + MF<T>::orow(lane, r);
        nv[i][r] = n < t0.N;
        cn[i][r] = tCN[nv[i][r] ? n : 0];
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (mv[j] && nv[i][r]) {
            const int64_t ad = cm[j] + cn[i][r];
            double v = alpha * double(acc[i][j][r]);
            if (beta != 0.0) v += beta * Cb[ad];
            Cb[ad] = v;
          }
        }
  }
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The two BF16 terms of x and y (x in the low halves).  v_cvt_pk_bf16_f32
// rounds to nearest even, as the integer form it replaced did for every float
// but NaN, which now stays one.
__device__ __forceinline__ void split_bf16x2(double x, double y, uint32_t &hi, uint32_t &lo) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  const f2 f{float(x), float(y)};
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, b2));
  const f2 r{f.x - __uint_as_float(hi << 16), f.y - __uint_as_float(hi & 0xFFFF0000u)};
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, b2));
}
__device__ __forceinline__ void split_bf16(double x, unsigned short &hi, unsigned short &lo) {
  uint32_t h, l;
  split_bf16x2(x, 0.0, h, l);
  hi = (unsigned short)h;
  lo = (unsigned short)l;
}

// ---- register-pipelined tiles of any size, layout and alignment ---------------
// The pipeline of k_dgemm in every form, with (32 FM) x (32 FN) tiles.  Each
// operand is loaded in aligned runs of k (V = 2 or 4, both operands), single
// elements with the lanes along k (V = 1) or along the rows (V = 0, so an
// operand contiguous along its rows coalesces).  Rows and columns past the
// block load its last one and are not stored, so only the k past the end has
// to be zeroed, in the last stages: in the steady state no load or store has a
// condition, and they sit between the MFMAs by schedule groups.
// FP64 (k order 4q + s): a stage of 128 x 128 is 1.87 us, 1.7 of it MFMA.
// 64 x 64: four times the units for products that leave CUs idle with the
// larger tile, two workgroups per CU.  Dense chain, first and last stage, from
// k_gemm / k_dgemm: chi = 1024 773 + 728 to 624 + 593 us (the matrix cores
// need 563 each), chi = 512 136 + 148 to 100 + 96, chi = 255 28 + 43 to 26.5 +
// 28.5.
// FP32 (natural k order, the bits of k_gemm): operands arrive as FP64, so a
// stage moves twice the bytes its MFMAs suggest; 128 x 128 1.13 us (0.82 of
// MFMA), 64 x 64 0.33 with several workgroups on the CU, 0.43 alone.  chi = 512
// 84 + 135 to 66 + 75 us, chi = 1024 596 + 539 to 380 + 350.  Stages of 32 k
// gained 15% where one workgroup has a CU to itself and lost 5-10% elsewhere.
// BF16x3 (bits of k_gemm3): the one wave of a SIMD also converts 32 elements a
// lane and stage, about as long as its 48 MFMAs; 128 x 128 1.4 us for 32 k
// (MFMA 0.32).  chi = 768 168 + 188 to 116 + 157 us, chi = 1024 343 + 289 to
// 235 + 210.  Spreading the conversions over the stage by schedule groups made
// 128 x 128 wait for its newest loads: 245 + 411 us.
// T: double, float, or unsigned short for the two BF16 terms.  An LDS row:
// the k of a stage; BF16x3 32 hi, then 32 lo terms (pitch 144 bytes).
template <typename T>
constexpr int kPipeBK = sizeof(T) == 2 ? 32 : DG_BK;
template <typename T>
constexpr int kPipePitch = sizeof(T) == 8 ? 18 : sizeof(T) == 4 ? 20 : 72;

// One operand: ROWS rows of a stage; SP: pre-split words instead of FP64.
template <typename T, int ROWS, int V, bool SP>
struct PipeLoader {
  using RT = std::conditional_t<SP, uint32_t, double>;
  static constexpr int KB = kPipeBK<T>;
  static constexpr int LK = V ? KB / (V ? V : 1) : DG_NT / (ROWS < 64 ? ROWS : 64);  // lanes along k
  static constexpr int RS = DG_NT / LK, NP = ROWS / RS, NE = V ? V : KB / LK, NK = V ? 1 : NE;
  static constexpr int NR = NP * NE;                                                 // elements of a thread
  static constexpr int NLD = NR / (V == 0 ? 1 : SP ? V : V == 4 ? 2 : V);            // loads
  static constexpr int NST = sizeof(T) == 8 ? (NE == 1 ? NR : NR / 2)                // LDS stores
                             : sizeof(T) == 4 ? NR : 2 * NR / (NE < 4 ? NE : 4);
  int64_t roff[NP];
  int64_t ko[2][NK];  // k offsets of the next two stages to load (slot = stage & 1)
  int lr, lc;         // first row; first k
  __device__ __forceinline__ void init(int tid, int row0, int R, const int64_t *__restrict__ tabR) {
    lc = V ? V * (tid % LK) : NE * (RS == 64 ? __builtin_amdgcn_readfirstlane(tid / RS) : tid / RS);
    lr = V ? tid / LK : tid % RS;
#pragma unroll
    for (int p = 0; p < NP; ++p) roff[p] = tabR[min(row0 + lr + RS * p, R - 1)];
  }
  __device__ __forceinline__ void fetch_k(int k0, int K, const int64_t *__restrict__ tabK, int slot) {
#pragma unroll
    for (int c = 0; c < NK; ++c) ko[slot][c] = tabK[min(k0 + lc + c, K - (V ? V : 1))];
  }
  __device__ __forceinline__ void load(const RT *__restrict__ base, RT (&r)[NR], int slot) const {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const RT *q = base + roff[p] + ko[slot][0];
      if constexpr (V == 0) {
#pragma unroll
        for (int c = 0; c < NK; ++c) r[NK * p + c] = (base + ko[slot][c])[roff[p]];
      } else if constexpr (V == 1) {
        r[p] = *q;
      } else if constexpr (SP) {
        const uint4 v = *reinterpret_cast<const uint4 *>(q);
        r[4 * p] = v.x;
        r[4 * p + 1] = v.y;
        r[4 * p + 2] = v.z;
        r[4 * p + 3] = v.w;
      } else {
#pragma unroll
        for (int c = 0; c < V; c += 2) {
          const double2 v = *reinterpret_cast<const double2 *>(q + c);
          r[V * p + c] = v.x;
          r[V * p + c + 1] = v.y;
        }
      }
    }
  }
  // Where the fragment reads want k: FP64 k = 4q + s in the lanes of quarter
  // q at MFMA s, FP32 k = 4s + q (the sums of k_gemm, to the last bit).
  static __device__ __forceinline__ int place(int k) { return sizeof(T) == 8 ? k : 4 * (k & 3) + (k >> 2); }
  // k0: first k of the stage (TAIL: its k past K are zeroed)
  template <bool TAIL>
  __device__ __forceinline__ void store(T *__restrict__ s, const RT (&r)[NR], int k0, int K) const {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      T *d = s + (lr + RS * p) * kPipePitch<T>;
      auto in = [&](int c) { return !TAIL || k0 + lc + c < K ? r[NE * p + c] : RT(0); };
      if constexpr (sizeof(T) == 2) {
        if constexpr (NE == 1) {
          uint32_t h = 0, l = 0;
          if constexpr (SP) {
            h = in(0);
            l = h >> 16;
          } else {
            split_bf16x2(in(0), 0.0, h, l);
          }
          d[lc] = T(h);
          d[KB + lc] = T(l);
        } else {
#pragma unroll
          for (int c = 0; c < NE; c += 4) {
            uint2 h, l;
            if constexpr (SP) {
              const uint32_t w0 = in(c), w1 = in(c + 1), w2 = in(c + 2), w3 = in(c + 3);
              h = uint2{(w0 & 0xFFFFu) | (w1 << 16), (w2 & 0xFFFFu) | (w3 << 16)};
              l = uint2{(w0 >> 16) | (w1 & 0xFFFF0000u), (w2 >> 16) | (w3 & 0xFFFF0000u)};
            } else {
              split_bf16x2(in(c), in(c + 1), h.x, l.x);
              split_bf16x2(in(c + 2), in(c + 3), h.y, l.y);
            }
            *reinterpret_cast<uint2 *>(d + lc + c) = h;
            *reinterpret_cast<uint2 *>(d + KB + lc + c) = l;
          }
        }
      } else if constexpr (sizeof(T) == 8 && NE > 1) {
#pragma unroll
        for (int c = 0; c < NE; c += 2) *reinterpret_cast<double2 *>(d + lc + c) = double2{in(c), in(c + 1)};
      } else {
#pragma unroll
        for (int c = 0; c < NE; ++c) d[place(lc + c)] = T(in(c));
      }
    }
  }
};

template <typename T, int F>
struct PipeFrag {  // one operand of a stage: F fragments x 4 k (BF16x3: 8 k, both terms)
  using Quad = std::conditional_t<sizeof(T) == 8, double2[2], std::conditional_t<sizeof(T) == 4, float4, bf16x8[2]>>;
  Quad x[F];
  __device__ __forceinline__ void read(const T *__restrict__ s, int row0, int lane) {
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const T *p = s + (row0 + j * 16 + (lane & 15)) * kPipePitch<T> + kPipeBK<T> / 4 * (lane >> 4);
      if constexpr (sizeof(T) == 8) {
        x[j][0] = *reinterpret_cast<const double2 *>(p);
        x[j][1] = *reinterpret_cast<const double2 *>(p + 2);
      } else if constexpr (sizeof(T) == 4) {
        x[j] = *reinterpret_cast<const float4 *>(p);
      } else {
        x[j][0] = *reinterpret_cast<const bf16x8 *>(p);
        x[j][1] = *reinterpret_cast<const bf16x8 *>(p + kPipeBK<T>);
      }
    }
  }
};

template <typename T, int FM, int FN, int VA, int VB, bool SP = false>
__global__ __launch_bounds__(DG_NT, FM * FN <= 4 ? 2 : 1) void k_pipe(
    const double *__restrict__ A, const double *__restrict__ B, double *__restrict__ C,
    const GemmTask *__restrict__ tasks, const WorkUnit *__restrict__ units, int nunits, const int64_t *__restrict__ tab,
    double alpha, double beta) {
  using M = MF<std::conditional_t<sizeof(T) == 2, float, T>>;
  using v4 = typename M::v4;
  constexpr int P = kPipePitch<T>, KB = kPipeBK<T>, BM = 32 * FM, BN = 32 * FN;
  constexpr int NM = sizeof(T) == 2 ? 3 * FM * FN / 4 : FM * FN;  // MFMAs of a quarter of a stage
  constexpr int NRD = (sizeof(T) == 4 ? 1 : 2) * (FM + FN);  // LDS reads of a stage
  using LA = PipeLoader<T, BM, VA, SP>;
  using LB = PipeLoader<T, BN, VB, SP>;
  __shared__ __align__(16) T As[2][BM * P];
  __shared__ __align__(16) T Bs[2][BN * P];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 16 * FM, wn = (wave >> 1) * 16 * FN;

  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    v4 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = v4{0, 0, 0, 0};

    for (int t = wu.tbeg; t < wu.tend; ++t) {
      const GemmTask tk = tasks[t];
      if (tk.K <= 0) continue;
      LA la;
      LB lb;
      la.init(tid, wu.m0, tk.M, tab + tk.tAM);
      lb.init(tid, wu.n0, tk.N, tab + tk.tBN);
      using RT = typename LA::RT;  // SP: the pointers are the split words, typed as FP64
      const RT *Ab = reinterpret_cast<const RT *>(A) + tk.a_off;
      const RT *Bb = reinterpret_cast<const RT *>(B) + tk.b_off;
      const int64_t *tAK = tab + tk.tAK;
      const int64_t *tBK = tab + tk.tBK;
      const int K = tk.K, S = (K + KB - 1) / KB;
      RT ra0[LA::NR], rb0[LB::NR], ra1[LA::NR], rb1[LB::NR];  // load register sets
#define ITX_PIPE_LOAD(st, ra, rb, slot)                   \
  {                                                       \
    la.load(Ab, ra, slot);                                \
    lb.load(Bb, rb, slot);                                \
    la.fetch_k(((st) + 2) * KB, K, tAK, slot);         \
    lb.fetch_k(((st) + 2) * KB, K, tBK, slot);         \
  }
#define ITX_PIPE_STORE(tail, st, ra, rb)                                  \
  {                                                                       \
    la.template store<tail>(As[(st) & 1], ra, (st) * KB, K);           \
    lb.template store<tail>(Bs[(st) & 1], rb, (st) * KB, K);           \
  }
      PipeFrag<T, FM> fa0, fa1;
      PipeFrag<T, FN> fb0, fb1;
      auto mfma = [&](const PipeFrag<T, FM> &fa, const PipeFrag<T, FN> &fb, int s) __attribute__((always_inline)) {
        if constexpr (sizeof(T) == 2) {  // a quarter of the fragments: the two cross terms, then hi * hi
#pragma unroll
          for (int e = 0; e < 3; ++e)
#pragma unroll
            for (int h = s * FM * FN / 4; h < (s + 1) * FM * FN / 4; ++h)
              acc[h / FM][h % FM] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  fb.x[h / FM][e == 1], fa.x[h % FM][e == 0], acc[h / FM][h % FM], 0, 0, 0);
        } else {
#pragma unroll
          for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j) acc[i][j] = M::mma(dg_k(fb.x[i], s), dg_k(fa.x[j], s), acc[i][j]);
        }
      };
      la.fetch_k(0, K, tAK, 0);
      lb.fetch_k(0, K, tBK, 0);
      la.fetch_k(KB, K, tAK, 1);
      lb.fetch_k(KB, K, tBK, 1);
      ITX_PIPE_LOAD(0, ra0, rb0, 0)
      if (S > 1) ITX_PIPE_LOAD(1, ra1, rb1, 1)
      __syncthreads();  // the previous task's LDS reads are done
      ITX_PIPE_STORE(true, 0, ra0, rb0)
      if (S > 2) ITX_PIPE_LOAD(2, ra0, rb0, 0)
      __syncthreads();
      fa0.read(As[0], wm, lane);
      fb0.read(Bs[0], wn, lane);
      if (S > 1) ITX_PIPE_STORE(true, 1, ra1, rb1)
      if (S > 3) ITX_PIPE_LOAD(3, ra1, rb1, 1)
      __syncthreads();
      // stage n: read stage n+1, store n+2, load n+4 around its MFMAs
#define ITX_PIPE_STEP(n, fa, fb, na, nb, ra, rb, slot)            \
  {                                                               \
    if ((n) + 1 < S) {                                            \
      na.read(As[((n) + 1) & 1], wm, lane);                       \
      nb.read(Bs[((n) + 1) & 1], wn, lane);                       \
    }                                                             \
    mfma(fa, fb, 0);                                              \
    __builtin_amdgcn_sched_barrier(0);                            \
    if ((n) + 2 < S) ITX_PIPE_STORE(true, (n) + 2, ra, rb)        \
    if ((n) + 4 < S) ITX_PIPE_LOAD((n) + 4, ra, rb, slot)         \
    __builtin_amdgcn_sched_barrier(0);                            \
    mfma(fa, fb, 1);                                              \
    mfma(fa, fb, 2);                                              \
    mfma(fa, fb, 3);                                              \
    __builtin_amdgcn_sched_barrier(0);                            \
    __syncthreads();                                              \
  }
      // steady state (n + 4 < S): no conditions, the other instructions
      // placed between the MFMAs
#define ITX_PIPE_BODY(n, fa, fb, na, nb, ra, rb, id)                                             \
  {                                                                                              \
    na.read(As[((n) + 1) & 1], wm, lane);                                                        \
    nb.read(Bs[((n) + 1) & 1], wn, lane);                                                        \
    mfma(fa, fb, 0);                                                                             \
    for (int g_ = 0; g_ < NM; ++g_) {                                                            \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, id);                                        \
      __builtin_amdgcn_sched_group_barrier(0x100, (NRD + NM - 1) / NM, id);                      \
    }                                                                                            \
    __builtin_amdgcn_sched_barrier(0);                                                           \
    ITX_PIPE_STORE(false, (n) + 2, ra, rb)                                                       \
    mfma(fa, fb, 1);                                                                             \
    for (int g_ = 0; g_ < NM; ++g_) {                                                            \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, id);                                        \
      __builtin_amdgcn_sched_group_barrier(0x200, (LA::NST + LB::NST + NM - 1) / NM, id);        \
    }                                                                                            \
    __builtin_amdgcn_sched_barrier(0);                                                           \
    ITX_PIPE_LOAD((n) + 4, ra, rb, id)                                                           \
    mfma(fa, fb, 2);                                                                             \
    for (int g_ = 0; g_ < NM; ++g_) {                                                            \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, id);                                        \
      __builtin_amdgcn_sched_group_barrier(0x006, 8, id);                                        \
      __builtin_amdgcn_sched_group_barrier(0x020, (LA::NLD + LB::NLD + 2 + NM - 1) / NM, id);    \
    }                                                                                            \
    __builtin_amdgcn_sched_barrier(0);                                                           \
    mfma(fa, fb, 3);                                                                             \
    __builtin_amdgcn_sched_barrier(0);                                                           \
    __syncthreads();                                                                             \
  }
      int n = 0;
      for (; n + 5 < S; n += 2) {
        ITX_PIPE_BODY(n, fa0, fb0, fa1, fb1, ra0, rb0, 0)
        ITX_PIPE_BODY(n + 1, fa1, fb1, fa0, fb0, ra1, rb1, 1)
      }
      for (; n + 1 < S; n += 2) {
        ITX_PIPE_STEP(n, fa0, fb0, fa1, fb1, ra0, rb0, 0)
        ITX_PIPE_STEP(n + 1, fa1, fb1, fa0, fb0, ra1, rb1, 1)
      }
      if (n < S) ITX_PIPE_STEP(n, fa0, fb0, fa1, fb1, ra0, rb0, 0)
#undef ITX_PIPE_BODY
#undef ITX_PIPE_STEP
#undef ITX_PIPE_STORE
#undef ITX_PIPE_LOAD
    }

    if (sizeof(T) == 8 && wu.slot >= 0) {  // partial tile of a split unit (C is the workspace)
      double *Pt = C + size_t(wu.slot) * (BM * BN);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < FM; ++j)
            Pt[(wn + i * 16 + M::orow(lane, r)) * BM + wm + j * 16 + (lane & 15)] = acc[i][j][r];
      continue;
    }
    const GemmTask t0 = tasks[wu.tbeg];
    const int64_t *tCM = tab + t0.tCM;
    const int64_t *tCN = tab + t0.tCN;
    double *Cb = C + t0.c_off;
    int64_t cm[FM], cn[FN][4];
#pragma unroll
    for (int j = 0; j < FM; ++j) cm[j] = tCM[min(wu.m0 + wm + j * 16 + (lane & 15), t0.M - 1)];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) cn[i][r] = tCN[min(wu.n0 + wn + i * 16 + M::orow(lane, r), t0.N - 1)];
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = wu.m0 + wm + j * 16 + (lane & 15), n = wu.n0 + wn + i * 16 + M::orow(lane, r);
          if (m < t0.M && n < t0.N) {
            const int64_t ad = cm[j] + cn[i][r];
            double v = alpha * double(acc[i][j][r]);
            if (beta != 0.0) v += beta * Cb[ad];
            Cb[ad] = v;
          }
        }
  }
}

// ---- BF16x3 form ----------------------------------------------------------
// Each FP64 operand value is rounded to FP32 and split into two BF16 terms
// x ~ hi + lo (hi = bf16(x), lo = bf16(x - hi): 16-17 significant bits);
// a product is formed from the three leading terms hi*hi + hi*lo + lo*hi on
// the BF16 MFMA (v_mfma_f32_16x16x32_bf16) with FP32 accumulation (the
// dropped lo*lo term is below 2^-16 relative).  LDS tiles are [row][k]
// with k contiguous so that a lane's 8 consecutive k of one row (its MFMA
// operand) are one 16-byte read; rows are padded to 80 bytes, which keeps
// the 16 rows read by a quarter-wave on distinct banks.
constexpr int BK3 = 32;        // K depth of one LDS stage = one bf16 MFMA
constexpr int LDK3 = BK3 + 8;  // bf16 elements per LDS row

// The pre-split operand format: y[i] = hi | lo << 16 of split_bf16(x[i]).
__global__ __launch_bounds__(256) void k_split_bf16(const double *__restrict__ x, uint32_t *__restrict__ y, size_t n) {
  for (size_t i = size_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += size_t(gridDim.x) * 256) {
    unsigned short h, l;
    split_bf16(x[i], h, l);
    y[i] = uint32_t(h) | (uint32_t(l) << 16);
  }
}

// With V = 4 (k-contiguous operands whose k runs come in aligned quads,
// checked when the plan is built) a lane loads four consecutive k of one
// row as two 16-byte loads and writes their hi and lo terms to LDS as one
// 8-byte store each.
// With SP the operand comes pre-split (itx_split_bf16): one 32-bit word per
// element, hi term in the low half and lo term in the high half, as
// split_bf16 forms them; the loader moves half the bytes and does no
// conversion (V = 4: one 16-byte load per quad).
template <int BR, bool KC, int NTH, int V = 1, bool SP = false>
struct TileLoader3 {
  static constexpr int PER = BR * BK3 / NTH;
  static_assert(PER >= 1, "tile too small for the thread count");
  static_assert(V == 1 || (KC && V == 4 && PER % V == 0), "vector loads need a k-contiguous operand");
  static constexpr int NV = PER / V;
  static constexpr int LK = BK3 / V;
  static constexpr int NK = KC ? 1 : PER;
  using RT = std::conditional_t<SP, uint32_t, double>;
  RT r[PER];
  bool rok[NV];
  int64_t roff[KC ? NV : 1];
  bool rv[KC ? NV : 1];
  int64_t ko[NK];
  bool kv[NK];
  int lr, lk;

  __device__ __forceinline__ void init(int tid, int row0, int R, const int64_t *__restrict__ tabR) {
    if constexpr (KC) {
      lk = (tid % LK) * V;
      lr = tid / LK;
#pragma unroll
      for (int p = 0; p < NV; ++p) {
        const int row = row0 + lr + (NTH / LK) * p;
        rv[p] = row < R;
        roff[p] = tabR[rv[p] ? row : 0];
      }
    } else {
      lr = tid % BR;
      lk = tid / BR;
      const int row = row0 + lr;
      rv[0] = row < R;
      roff[0] = tabR[rv[0] ? row : 0];
    }
  }
  __device__ __forceinline__ void fetch_k(int k0, int K, const int64_t *__restrict__ tabK) {
#pragma unroll
    for (int q = 0; q < NK; ++q) {
      const int k = k0 + lk + (KC ? 0 : (NTH / BR) * q);
      kv[q] = k < K;
      ko[q] = tabK[kv[q] ? k : 0];
    }
  }
  __device__ __forceinline__ void load(const void *__restrict__ base_) {
    const RT *__restrict__ base = static_cast<const RT *>(base_);
#pragma unroll
    for (int p = 0; p < NV; ++p) {
      const bool ok = KC ? (kv[0] && rv[p]) : (kv[p] && rv[0]);
      const int64_t off = (KC ? roff[p] + ko[0] : roff[0] + ko[p]);
      if constexpr (V == 4 && SP) {
        const uint4 v = *reinterpret_cast<const uint4 *>(base + (ok ? off : 0));
        r[4 * p] = v.x;
        r[4 * p + 1] = v.y;
        r[4 * p + 2] = v.z;
        r[4 * p + 3] = v.w;
      } else if constexpr (V == 4) {
        const double2 *q = reinterpret_cast<const double2 *>(base + (ok ? off : 0));
        const double2 v0 = q[0], v1 = q[1];
        r[4 * p] = v0.x;
        r[4 * p + 1] = v0.y;
        r[4 * p + 2] = v1.x;
        r[4 * p + 3] = v1.y;
      } else {
        r[p] = base[ok ? off : 0];
      }
      rok[p] = ok;
    }
  }
  __device__ __forceinline__ void store(unsigned short *__restrict__ sh, unsigned short *__restrict__ sl) const {
    if constexpr (V == 4 && SP) {
#pragma unroll
      for (int p = 0; p < NV; ++p) {
        const int idx = (lr + (NTH / LK) * p) * LDK3 + lk;
        const uint32_t z = rok[p] ? 0xFFFFFFFFu : 0u;
        const uint32_t w0 = r[4 * p] & z, w1 = r[4 * p + 1] & z, w2 = r[4 * p + 2] & z, w3 = r[4 * p + 3] & z;
        *reinterpret_cast<uint2 *>(&sh[idx]) = uint2{(w0 & 0xFFFFu) | (w1 << 16), (w2 & 0xFFFFu) | (w3 << 16)};
        *reinterpret_cast<uint2 *>(&sl[idx]) =
            uint2{(w0 >> 16) | (w1 & 0xFFFF0000u), (w2 >> 16) | (w3 & 0xFFFF0000u)};
      }
    } else if constexpr (SP) {
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int idx = KC ? (lr + (NTH / BK3) * p) * LDK3 + lk : lr * LDK3 + lk + (NTH / BR) * p;
        const uint32_t w = rok[p] ? r[p] : 0u;
        sh[idx] = (unsigned short)(w & 0xFFFFu);
        sl[idx] = (unsigned short)(w >> 16);
      }
    } else if constexpr (V == 4) {
#pragma unroll
      for (int p = 0; p < NV; ++p) {
        const int idx = (lr + (NTH / LK) * p) * LDK3 + lk;
        uint2 h{0, 0}, l{0, 0};
        if (rok[p]) {
          split_bf16x2(r[4 * p], r[4 * p + 1], h.x, l.x);
          split_bf16x2(r[4 * p + 2], r[4 * p + 3], h.y, l.y);
        }
        *reinterpret_cast<uint2 *>(&sh[idx]) = h;
        *reinterpret_cast<uint2 *>(&sl[idx]) = l;
      }
    } else {
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int idx = KC ? (lr + (NTH / BK3) * p) * LDK3 + lk : lr * LDK3 + lk + (NTH / BR) * p;
        unsigned short h = 0, l = 0;
        if (rok[p]) split_bf16(r[p], h, l);
        sh[idx] = h;
        sl[idx] = l;
      }
    }
  }
};

// SP: both operands pre-split (their pointers are the split words, typed
// as the other forms' FP64 operands)
template <int BM, int BN, int GM, int GN, bool AKC, bool BKC, int V, bool SP = false>
__global__ __launch_bounds__(64 * GM * GN) void k_gemm3(const double *__restrict__ A, const double *__restrict__ B,
                                                        double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                        const WorkUnit *__restrict__ units, int nunits,
                                                        const int64_t *__restrict__ tab, double alpha, double beta) {
  constexpr int NTH = 64 * GM * GN;
  typedef float v4 __attribute__((ext_vector_type(4)));
  using LA = TileLoader3<BM, AKC, NTH, V, SP>;
  using LB = TileLoader3<BN, BKC, NTH, V, SP>;
  constexpr int WM = BM / GM, WN = BN / GN, FM = WM / 16, FN = WN / 16;
  static_assert(FM >= 1 && FN >= 1, "wave tile below one MFMA fragment");
  __shared__ __align__(16) unsigned short Ah[2][BM * LDK3], Al[2][BM * LDK3];
  __shared__ __align__(16) unsigned short Bh[2][BN * LDK3], Bl[2][BN * LDK3];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % GM, wn = wave / GM;

  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    v4 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = v4{0, 0, 0, 0};

    for (int t = wu.tbeg; t < wu.tend; ++t) {
      const GemmTask tk = tasks[t];
      if (tk.K <= 0) continue;
      LA la;
      LB lb;
      la.init(tid, wu.m0, tk.M, tab + tk.tAM);
      lb.init(tid, wu.n0, tk.N, tab + tk.tBN);
      const void *Ab = SP ? static_cast<const void *>(reinterpret_cast<const uint32_t *>(A) + tk.a_off)
                          : static_cast<const void *>(A + tk.a_off);
      const void *Bb = SP ? static_cast<const void *>(reinterpret_cast<const uint32_t *>(B) + tk.b_off)
                          : static_cast<const void *>(B + tk.b_off);
      const int64_t *tAK = tab + tk.tAK;
      const int64_t *tBK = tab + tk.tBK;
      la.fetch_k(0, tk.K, tAK);
      lb.fetch_k(0, tk.K, tBK);
      la.load(Ab);
      lb.load(Bb);
      la.fetch_k(BK3, tk.K, tAK);
      lb.fetch_k(BK3, tk.K, tBK);
      la.store(Ah[0], Al[0]);
      lb.store(Bh[0], Bl[0]);
      __syncthreads();
      int cur = 0;
      for (int k0 = 0; k0 < tk.K; k0 += BK3) {
        const bool nxt = k0 + BK3 < tk.K;
        if (nxt) {
          la.load(Ab);
          lb.load(Bb);
          la.fetch_k(k0 + 2 * BK3, tk.K, tAK);
          lb.fetch_k(k0 + 2 * BK3, tk.K, tBK);
        }
        const int k8 = 8 * (lane >> 4);
        bf16x8 ah[FM], al[FM], bh[FN], bl[FN];
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          const int m = wm * WM + j * 16 + (lane & 15);
          ah[j] = *reinterpret_cast<const bf16x8 *>(&Ah[cur][m * LDK3 + k8]);
          al[j] = *reinterpret_cast<const bf16x8 *>(&Al[cur][m * LDK3 + k8]);
        }
#pragma unroll
        for (int i = 0; i < FN; ++i) {
          const int n = wn * WN + i * 16 + (lane & 15);
          bh[i] = *reinterpret_cast<const bf16x8 *>(&Bh[cur][n * LDK3 + k8]);
          bl[i] = *reinterpret_cast<const bf16x8 *>(&Bl[cur][n * LDK3 + k8]);
        }
        // D^T tile as in k_gemm; the two cross terms first, then hi*hi
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
          for (int j = 0; j < FM; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[i], al[j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[i], ah[j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[i], ah[j], acc[i][j], 0, 0, 0);
          }
        if (nxt) {
          la.store(Ah[cur ^ 1], Al[cur ^ 1]);
          lb.store(Bh[cur ^ 1], Bl[cur ^ 1]);
        }
        __syncthreads();
        cur ^= 1;
      }
    }

    const GemmTask t0 = tasks[wu.tbeg];
    const int64_t *tCM = tab + t0.tCM;
    const int64_t *tCN = tab + t0.tCN;
    double *Cb = C + t0.c_off;
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = wu.m0 + wm * WM + j * 16 + (lane & 15);
      if (m >= t0.M) continue;
      const int64_t cm = tCM[m];
#pragma unroll
      for (int i = 0; i < FN; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = wu.n0 + wn * WN + i * 16 + 4 * (lane >> 4) + r;
          if (n < t0.N) {
            const int64_t ad = cm + tCN[n];
            double v = alpha * double(acc[i][j][r]);
            if (beta != 0.0) v += beta * Cb[ad];
            Cb[ad] = v;
          }
        }
      }
    }
  }
}

// Skinny contractions (N <= 32 and K <= 64 for every task, e.g. the
// MPO-tensor stages of H*psi): HBM-bound, on the FP64 matrix cores in every
// form.  Same task/unit/table format as k_gemm.  A unit is 256 rows of one C
// block; each of its four waves takes 64 rows as four 16 x 16 MFMA row
// groups.  A lane loads the operands of its own fragment positions straight
// from memory (16 rows x 4 k: with A contiguous along k in runs of 4, or
// along m, a load instruction covers whole 128-byte lines) and the D^T tile
// stores 16 consecutive m per column, the four row groups of a column back
// to back.  No LDS and no barrier; 4 x S independent loads of A per lane are
// in flight, S = 1, 3 or 5 (SK_KS) slots of 4 k by what is left of a task: with
// five throughout, 500000 x 17 took 26 us for K = 1 (now 17.5) and 26 for K = 4
// (now 22), and ten blocks of some 10000 x 16 with three tasks of K <= 2 24 us
// (now 11).
// One task per unit with K <= 4 KS is straight-line code, the k offsets and
// B's fragments outside any loop (with the task and k loops around them the
// registers allowed two waves per SIMD when this was first measured: 104
// against 84 us at chi = 1024).
// K = N = 20 (the dense Heisenberg MPO pair), chi = 32, 255, 768, 1024: 6,
// 7, 32 and 75 us (84 before units of one block went by eighths to the XCDs);
// one thread per row with B in LDS, the form before this one, was bound by its
// K x N LDS reads and column tests: 22, 26, 84 and 115 us.  Stores past the
// caches make this kernel faster at chi = 1024 (54 us) and the next stage,
// which reads C back, slower by more (the chain 1514 against 1495 us).
constexpr int SK_ROWS = 256, SK_N = 32, SK_K = 64;
constexpr int SK_KS = 5;  // most k slots (of 4) loaded together: K = 20 in one chunk
constexpr int SK_G = 4;   // 16-row groups of a wave

// NB 16-column groups: 1 (N <= 16) or 2; KS: one task per unit, K <= 4 KS (0:
// any)
template <int NB, int KS>
__global__ __launch_bounds__(SK_ROWS, 3) void k_skinny(const double *__restrict__ A, const double *__restrict__ B,
                                                       double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                       const WorkUnit *__restrict__ units, int nunits,
                                                       const int64_t *__restrict__ tab, double alpha, double beta) {
  using v4 = MF<double>::v4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, q4 = lane >> 4;
  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    const GemmTask t0 = tasks[wu.tbeg];
    const int mb = wu.m0 + 16 * SK_G * wave;
    if (mb >= t0.M) continue;  // wave-uniform
    int mr[SK_G];  // rows past the block repeat its last row and are not stored
#pragma unroll
    for (int g = 0; g < SK_G; ++g) mr[g] = min(mb + 16 * g + r16, t0.M - 1);
    v4 acc[NB][SK_G];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int g = 0; g < SK_G; ++g) acc[i][g] = v4{0, 0, 0, 0};
    // 4 S k of one task: loads from clamped positions, zeroed where k
    // or the column is past the end, so no branch separates them
    auto chunk = [&](const GemmTask &tk, int k0, auto slots) __attribute__((always_inline)) {
      constexpr int S = decltype(slots)::value;
      double a[S][SK_G], b[S][NB];
      int64_t ka[S];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int k = k0 + 4 * s + q4;
        const bool kv = k < tk.K;
        ka[s] = tab[tk.tAK + (kv ? k : 0)];
        const int64_t kb = tab[tk.tBK + (kv ? k : 0)];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const bool nv = 16 * i + r16 < tk.N;
          const double x = B[tk.b_off + kb + tab[tk.tBN + (nv ? 16 * i + r16 : 0)]];
          b[s][i] = (kv && nv) ? x : 0.0;
        }
      }
#pragma unroll
      for (int g = 0; g < SK_G; ++g) {
        const double *Ar = A + tk.a_off + tab[tk.tAM + mr[g]];
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const double x = Ar[ka[s]];
          a[s][g] = k0 + 4 * s + q4 < tk.K ? x : 0.0;
        }
      }
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int g = 0; g < SK_G; ++g) acc[i][g] = MF<double>::mma(b[s][i], a[s][g], acc[i][g]);
    };
    if constexpr (KS > 0) {
      if (t0.K > 0) chunk(t0, 0, std::integral_constant<int, KS>{});
    } else {
      for (int t = wu.tbeg; t < wu.tend; ++t) {
        const GemmTask tk = tasks[t];
        int k0 = 0;
        for (; tk.K - k0 > 12; k0 += 4 * SK_KS) chunk(tk, k0, std::integral_constant<int, SK_KS>{});
        if (tk.K - k0 > 4)
          chunk(tk, k0, std::integral_constant<int, 3>{});
        else if (tk.K > k0)
          chunk(tk, k0, std::integral_constant<int, 1>{});
      }
    }
    int64_t cm[SK_G];
#pragma unroll
    for (int g = 0; g < SK_G; ++g) cm[g] = t0.c_off + tab[t0.tCM + mr[g]];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = 16 * i + MF<double>::orow(lane, r);
        if (n >= t0.N) continue;
        const int64_t cn = tab[t0.tCN + n];
#pragma unroll
        for (int g = 0; g < SK_G; ++g) {
          if (mb + 16 * g + r16 >= t0.M) continue;
          double *cp = C + cm[g] + cn;
          double v = alpha * acc[i][g][r];
          if (beta != 0.0) v += beta * (*cp);
          *cp = v;
        }
      }
  }
}

// The skinny path when every task has K <= 8 and N <= 8 (the block-pair
// tasks of a block-sparse MPO stage: site and MPO-link blocks of a few
// rows): a unit then sums many tiny tasks, and the per-task load round trip
// and LDS barriers of k_skinny dominate.  Here the B tiles of as many tasks
// as fit are staged in LDS at once (rows stacked), and the A elements of
// SKQ_G tasks are loaded together before any is used, those of the first
// before B is staged.  Tasks in order, k in order.  Bound by the trips of a
// unit (unit, tasks, tables, A and B, C) over two rounds of units: the MPO
// stage of the chi = 1024 block-sparse chain 19.3 us for 26 MB.
// Each thread computes two rows, SK_ROWS apart (units of 2 * SK_ROWS rows):
// the per-unit task reads, B staging and barriers are shared by twice the
// rows, and a thread has the loads of two rows in flight.
constexpr int SKQ_K = 8, SKQ_N = 8, SKQ_G = 2, SKQ_R = 2;

__global__ __launch_bounds__(SK_ROWS) void k_skinny_q(const double *__restrict__ A, const double *__restrict__ B,
                                                      double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                      const WorkUnit *__restrict__ units, int nunits,
                                                      const int64_t *__restrict__ tab, double alpha, double beta) {
  __shared__ double Bs[SK_K * SKQ_N];
  const int tid = threadIdx.x;
  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    const GemmTask t0 = tasks[wu.tbeg];
    const int N = t0.N, M = t0.M;
    int mr[SKQ_R];
    int64_t cr[SKQ_R];
    bool in[SKQ_R];
#pragma unroll
    for (int h = 0; h < SKQ_R; ++h) {
      mr[h] = wu.m0 + tid + h * SK_ROWS;
      in[h] = mr[h] < M;
      cr[h] = t0.c_off + tab[t0.tCM + min(mr[h], M - 1)];
    }
    double acc[SKQ_R][SKQ_N];
#pragma unroll
    for (int h = 0; h < SKQ_R; ++h)
#pragma unroll
      for (int n = 0; n < SKQ_N; ++n) acc[h][n] = 0.0;
    for (int tc = wu.tbeg; tc < wu.tend;) {
      // the next tasks whose stacked B rows fit the LDS tile
      int te = tc, kt = 0;
      while (te < wu.tend && kt + tasks[te].K <= SK_K) kt += tasks[te++].K;
      double av[SKQ_R][SKQ_G][SKQ_K];
      int kk[SKQ_G];
      auto fetch = [&](int t) {
#pragma unroll
        for (int q = 0; q < SKQ_G; ++q) {
          kk[q] = 0;
          if (t + q < te) {
            const GemmTask tk = tasks[t + q];
            kk[q] = tk.K;
            const int64_t *tAK = tab + tk.tAK;
#pragma unroll
            for (int h = 0; h < SKQ_R; ++h) {
              const double *Ar = A + tk.a_off + tab[tk.tAM + min(mr[h], M - 1)];
#pragma unroll
              for (int j = 0; j < SKQ_K; ++j) av[h][q][j] = (j < tk.K && in[h]) ? Ar[tAK[j]] : 0.0;
            }
          }
        }
      };
      fetch(tc);  // on its way while B is staged
      lds_barrier();  // the previous chunk's B rows are no longer read
      for (int t = tc, kb = 0; t < te; ++t) {
        const GemmTask tk = tasks[t];
        for (int x = tid; x < tk.K * N; x += SK_ROWS) {
          const int k = x / N, n = x - k * N;
          Bs[(kb + k) * SKQ_N + n] = B[tk.b_off + tab[tk.tBK + k] + tab[tk.tBN + n]];
        }
        kb += tk.K;
      }
      lds_barrier();
      for (int t = tc, kb = 0; t < te;) {
#pragma unroll
        for (int q = 0; q < SKQ_G; ++q) {
#pragma unroll
          for (int j = 0; j < SKQ_K; ++j) {
            if (j < kk[q]) {
#pragma unroll
              for (int n = 0; n < SKQ_N; ++n)
                if (n < N) {
                  const double bv = Bs[(kb + j) * SKQ_N + n];
#pragma unroll
                  for (int h = 0; h < SKQ_R; ++h) acc[h][n] += av[h][q][j] * bv;
                }
            }
          }
          kb += kk[q];
        }
        t += SKQ_G;
        if (t < te) fetch(t);
      }
      tc = te;
    }
#pragma unroll
    for (int h = 0; h < SKQ_R; ++h) {
      if (in[h]) {
        double *Cm = C + cr[h];
        const int64_t *tCN = tab + t0.tCN;
#pragma unroll
        for (int n = 0; n < SKQ_N; ++n) {
          if (n < N) {
            double v = alpha * acc[h][n];
            if (beta != 0.0) v += beta * Cm[tCN[n]];
            Cm[tCN[n]] = v;
          }
        }
      }
    }
  }
}

// Small-block contractions (C blocks of a few thousand elements: the QN
// blocks of DMRG at moderate bond dimension).  Latency-bound: what counts is
// the number of dependent trips through memory of a unit, a 64 x 32 tile of
// one C block.  FP64 form, on the matrix cores straight from memory: a wave
// loads the fragments of 32 x 32 outputs for 16 k at once (rows over 16
// lanes, 4 k over the lane quarters) while it multiplies the previous 16, and
// the eight waves share a unit's k: with up to 32 rows each takes every eighth
// task (or, with fewer than eight tasks, every eighth 16 k of each), above
// that four waves per half of the rows.  The waves' sums meet in LDS once.
// Staging both tiles in LDS for VALU arithmetic, the form before this one,
// made two barriers and three such trips per 64 k and task; the last stage of
// the dense chi = 32 chain (one 128 x 32 block, K = 160) took 31 us with its
// reduction pass.
// Same task/unit/table format as k_gemm.
constexpr int SM_M = 64, SM_N = 32, SM_K = 64, SM_T = 256;
constexpr int SMD_W = 8, SMD_T = 64 * SMD_W;  // waves of the FP64 form
constexpr int SMD_P = 17;                     // its LDS row pitch

// One operand's 32 rows (or columns) x 16 k of a wave.  Contiguous along k
// (KC): lanes walk k, four rows per load (with lanes over rows each load
// would touch 64 separate segments, which the address unit takes one by one:
// 15 us for the chi = 32 block against 5), and the wave's own LDS buffer turns
// them into fragments; else lanes walk the rows and the loads are fragments.
template <bool KC>
struct SmallOperand {
  static constexpr int NR = KC ? 8 : 2;  // rows of a lane
  const double *row[NR];
  double x[8] = {};
  // rows: first row, last valid row; tab: its row offsets
  __device__ __forceinline__ void init(const double *base, int row0, int last, const int64_t *__restrict__ tab, int lane) {
#pragma unroll
    for (int p = 0; p < NR; ++p) {
      const int r = KC ? 4 * p + (lane >> 4) : 16 * p + (lane & 15);
      row[p] = base + tab[min(row0 + r, last)];
    }
  }
  // two: the second group of 16 rows is in use
  __device__ __forceinline__ void load(int k0, int K, const int64_t *__restrict__ tab, bool two, int lane) {
    if constexpr (KC) {
      const int64_t ko = tab[min(k0 + (lane & 15), K - 1)];
#pragma unroll
      for (int p = 0; p < 4; ++p) x[p] = row[p][ko];
      if (two) {
#pragma unroll
        for (int p = 4; p < 8; ++p) x[p] = row[p][ko];
      }
    } else {
      int64_t ko[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) ko[s] = tab[min(k0 + 4 * s + (lane >> 4), K - 1)];
#pragma unroll
      for (int s = 0; s < 4; ++s) x[2 * s] = row[0][ko[s]];
      if (two) {
#pragma unroll
        for (int s = 0; s < 4; ++s) x[2 * s + 1] = row[1][ko[s]];
      }
    }
  }
  // f[s][g]: fragment of k slot s, row group g
  __device__ __forceinline__ void fragments(double (&f)[4][2], double *buf, int lane) const {
    if constexpr (KC) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int p = 0; p < 8; ++p) buf[(4 * p + (lane >> 4)) * SMD_P + (lane & 15)] = x[p];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int g = 0; g < 2; ++g) f[s][g] = buf[(16 * g + (lane & 15)) * SMD_P + 4 * s + (lane >> 4)];
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int g = 0; g < 2; ++g) f[s][g] = x[2 * s + g];
    }
  }
};

template <bool AKC, bool BKC>
__global__ __launch_bounds__(SMD_T) void k_small(const double *__restrict__ A, const double *__restrict__ B,
                                                 double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                 const WorkUnit *__restrict__ units, int nunits,
                                                 const int64_t *__restrict__ tab, double alpha, double beta) {
  using v4 = MF<double>::v4;
  constexpr int BUF = 32 * SMD_P;
  __shared__ double lds[SMD_W * 2 * BUF];  // operand buffers of the waves, then their sums
  static_assert(2 * BUF >= 16 * 64, "room for the sums");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, q4 = lane >> 4;
  double *bufA = lds + wave * 2 * BUF, *bufB = bufA + BUF;
  double(*part)[16][64] = reinterpret_cast<double(*)[16][64]>(lds);
  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    const GemmTask t0 = tasks[wu.tbeg];
    // the unit's end: its tile (pad: rows | columns << 8) inside the block
    const int mend = min(t0.M, wu.m0 + (wu.pad & 255)), nend = min(t0.N, wu.n0 + (wu.pad >> 8));
    const bool tall = mend - wu.m0 > 32;
    const int mh = tall ? wave & 1 : 0, ks = tall ? wave >> 1 : wave, nks = tall ? SMD_W / 2 : SMD_W;
    const int m0 = wu.m0 + 32 * mh;
    const bool two_m = mend - m0 > 16, two_n = nend - wu.n0 > 16;
    v4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < 2; ++g) acc[i][g] = v4{0, 0, 0, 0};
    // the table entries of the results, long before they are needed
    const int fr = tall ? ks : wave >> 1;  // the fragment this wave finishes
    const int64_t cm = tab[t0.tCM + min(m0 + 16 * (fr & 1) + r16, t0.M - 1)];
    int64_t cn[4];
#pragma unroll
    for (int h = 0; h < 4; ++h)
      cn[h] = tab[t0.tCN + min(wu.n0 + 16 * (fr >> 1) + MF<double>::orow(lane, tall ? h : 2 * (wave & 1) + (h & 1)),
                               t0.N - 1)];
    const bool share = wu.tend - wu.tbeg < nks;  // few tasks: share each one's k
    const int kb = share ? 16 * ks : 0, kd = share ? 16 * nks : 16;
    for (int t = share ? wu.tbeg : wu.tbeg + ks; t < wu.tend; t += share ? 1 : nks) {
      const GemmTask tk = tasks[t];
      if (kb >= tk.K) continue;
      // rows past the block repeat its last one, k past the end is zeroed
      SmallOperand<AKC> oa;
      SmallOperand<BKC> ob;
      oa.init(A + tk.a_off, m0, t0.M - 1, tab + tk.tAM, lane);
      ob.init(B + tk.b_off, wu.n0, t0.N - 1, tab + tk.tBN, lane);
      oa.load(kb, tk.K, tab + tk.tAK, two_m, lane);
      ob.load(kb, tk.K, tab + tk.tBK, two_n, lane);
      for (int k0 = kb; k0 < tk.K; k0 += kd) {
        double a[4][2], b[4][2];
        oa.fragments(a, bufA, lane);
        ob.fragments(b, bufB, lane);
        if (k0 + kd < tk.K) {
          oa.load(k0 + kd, tk.K, tab + tk.tAK, two_m, lane);
          ob.load(k0 + kd, tk.K, tab + tk.tBK, two_n, lane);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          if (k0 + 4 * s >= tk.K) break;  // uniform
          const bool kv = k0 + 4 * s + q4 < tk.K;
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            a[s][g] = kv ? a[s][g] : 0.0;
            b[s][g] = kv ? b[s][g] : 0.0;
          }
          acc[0][0] = MF<double>::mma(b[s][0], a[s][0], acc[0][0]);
          if (two_m) acc[0][1] = MF<double>::mma(b[s][0], a[s][1], acc[0][1]);
          if (two_n) acc[1][0] = MF<double>::mma(b[s][1], a[s][0], acc[1][0]);
          if (two_m && two_n) acc[1][1] = MF<double>::mma(b[s][1], a[s][1], acc[1][1]);
        }
      }
    }
    // sums of the waves of one half of the rows, each wave a part of them
    __syncthreads();  // every wave is done with its buffers
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wave][(2 * i + g) * 4 + r][lane] = acc[i][g][r];
    __syncthreads();
    // tall: wave (ks, mh) finishes fragment ks of its half; else the wave pair
    // (2 f, 2 f + 1) the two halves of fragment f
    const int ig = fr, i = ig >> 1, g = ig & 1;
    const int m = m0 + 16 * g + r16;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int r = tall ? h : 2 * (wave & 1) + (h & 1);
      if (!tall && h > 1) break;
      double v = 0.0;
      if (tall) {
#pragma unroll
        for (int w = 0; w < SMD_W / 2; ++w) v += part[mh + 2 * w][ig * 4 + r][lane];
      } else {
#pragma unroll
        for (int w = 0; w < SMD_W; ++w) v += part[w][ig * 4 + r][lane];
      }
      const int n = wu.n0 + 16 * i + MF<double>::orow(lane, r);
      if (m >= mend || n >= nend) continue;
      if (wu.slot >= 0) {  // partial tile of a split unit (C is the workspace)
        C[size_t(wu.slot) * (SM_M * SM_N) + size_t(n - wu.n0) * SM_M + (m - wu.m0)] = v;
      } else {
        double *cp = C + t0.c_off + cm + cn[h];
        v *= alpha;
        if (beta != 0.0) v += beta * (*cp);
        *cp = v;
      }
    }
    __syncthreads();  // the sums are read before the next unit's operands
  }
}

// Small-block contractions on the matrix cores: the FP32 and BF16x3 forms
// of the small-block path (same 64 x 32 unit tiles, task/unit/table format,
// split units and partial-tile layout as k_small).  Each k chunk of the A
// and B tiles is staged in LDS zero-padded to the MFMA depth (and to the
// full tile: rows and columns outside the block are zeros, so the padded
// fragments add nothing); wave w computes rows 16w..16w+15 of the tile as
// two 16 x 16 MFMA fragments.
// FP32: operands rounded to FP32 at staging, v_mfma_f32_16x16x4f32.
constexpr int SMF_LDA = SM_M + 17, SMF_LDB = SM_N + 17;  // odd pitches: k-strided staging hits distinct banks

template <bool AKC, bool BKC>
__global__ __launch_bounds__(SM_T) void k_small_f32(const double *__restrict__ A, const double *__restrict__ B,
                                                    double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                    const WorkUnit *__restrict__ units, int nunits,
                                                    const int64_t *__restrict__ tab, double alpha, double beta) {
  typedef float v4 __attribute__((ext_vector_type(4)));
  __shared__ float As[SM_K * SMF_LDA];
  __shared__ float Bs[SM_K * SMF_LDB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    v4 acc[2] = {v4{0, 0, 0, 0}, v4{0, 0, 0, 0}};
    for (int t = wu.tbeg; t < wu.tend; ++t) {
      const GemmTask tk = tasks[t];
      const int rows = min(SM_M, tk.M - wu.m0), cols = min(SM_N, tk.N - wu.n0);
      for (int k0 = 0; k0 < tk.K; k0 += SM_K) {
        const int kc = min(SM_K, tk.K - k0), kcp = (kc + 3) & ~3;
        __syncthreads();  // the previous chunk's tiles are no longer read
        {
          const int lead = AKC ? kcp : SM_M;
          for (int e = tid; e < SM_M * kcp; e += SM_T) {
            const int q = e / lead, r = e - q * lead;
            const int m = AKC ? q : r, k = AKC ? r : q;
            float v = 0.f;
            if (m < rows && k < kc) v = float(A[tk.a_off + tab[tk.tAM + wu.m0 + m] + tab[tk.tAK + k0 + k]]);
            As[k * SMF_LDA + m] = v;
          }
        }
        {
          const int lead = BKC ? kcp : SM_N;
          for (int e = tid; e < SM_N * kcp; e += SM_T) {
            const int q = e / lead, r = e - q * lead;
            const int n = BKC ? q : r, k = BKC ? r : q;
            float v = 0.f;
            if (n < cols && k < kc) v = float(B[tk.b_off + tab[tk.tBK + k0 + k] + tab[tk.tBN + wu.n0 + n]]);
            Bs[k * SMF_LDB + n] = v;
          }
        }
        __syncthreads();
        const int kl = lane >> 4, ml = 16 * wave + (lane & 15);
        for (int kk = 0; kk < kcp; kk += 4) {
          const float a = As[(kk + kl) * SMF_LDA + ml];
          const float b0 = Bs[(kk + kl) * SMF_LDB + (lane & 15)];
          const float b1 = Bs[(kk + kl) * SMF_LDB + 16 + (lane & 15)];
          // D^T fragments: MFMA rows run over n, columns over m
          acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(b0, a, acc[0], 0, 0, 0);
          acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(b1, a, acc[1], 0, 0, 0);
        }
      }
    }
    const int ml = 16 * wave + (lane & 15);
    if (wu.slot >= 0) {  // partial tile of a split unit (C is the workspace)
      double *P = C + size_t(wu.slot) * (SM_M * SM_N);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) P[(16 * i + 4 * (lane >> 4) + r) * SM_M + ml] = double(acc[i][r]);
      continue;
    }
    const GemmTask t0 = tasks[wu.tbeg];
    const int m = wu.m0 + ml;
    if (m < t0.M) {
      double *Cm = C + t0.c_off + tab[t0.tCM + m];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = wu.n0 + 16 * i + 4 * (lane >> 4) + r;
          if (n < t0.N) {
            double *cp = Cm + tab[t0.tCN + n];
            double v = alpha * double(acc[i][r]);
            if (beta != 0.0) v += beta * (*cp);
            *cp = v;
          }
        }
    }
  }
}

// BF16x3: each operand value split at staging into x ~ hi + lo (the split
// of k_gemm3), tiles [row][k] with k contiguous so that a lane's 8
// consecutive k are one 16-byte LDS read; hi*lo + lo*hi + hi*hi on
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation.  k chunks are padded to
// the MFMA depth of 32.
constexpr int SM3_LD = SM_K + 8;  // bf16 elements per LDS row (16-byte aligned rows)

template <bool AKC, bool BKC>
__global__ __launch_bounds__(SM_T) void k_small_bf16x3(const double *__restrict__ A, const double *__restrict__ B,
                                                       double *__restrict__ C, const GemmTask *__restrict__ tasks,
                                                       const WorkUnit *__restrict__ units, int nunits,
                                                       const int64_t *__restrict__ tab, double alpha,
                                                       double beta) {
  typedef float v4 __attribute__((ext_vector_type(4)));
  __shared__ __align__(16) unsigned short Ah[SM_M * SM3_LD], Al[SM_M * SM3_LD];
  __shared__ __align__(16) unsigned short Bh[SM_N * SM3_LD], Bl[SM_N * SM3_LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    const WorkUnit wu = units[u];
    v4 acc[2] = {v4{0, 0, 0, 0}, v4{0, 0, 0, 0}};
    for (int t = wu.tbeg; t < wu.tend; ++t) {
      const GemmTask tk = tasks[t];
      const int rows = min(SM_M, tk.M - wu.m0), cols = min(SM_N, tk.N - wu.n0);
      for (int k0 = 0; k0 < tk.K; k0 += SM_K) {
        const int kc = min(SM_K, tk.K - k0), kcp = (kc + 31) & ~31;
        __syncthreads();
        {
          const int lead = AKC ? kcp : SM_M;
          for (int e = tid; e < SM_M * kcp; e += SM_T) {
            const int q = e / lead, r = e - q * lead;
            const int m = AKC ? q : r, k = AKC ? r : q;
            unsigned short h = 0, l = 0;
            if (m < rows && k < kc) split_bf16(A[tk.a_off + tab[tk.tAM + wu.m0 + m] + tab[tk.tAK + k0 + k]], h, l);
            Ah[m * SM3_LD + k] = h;
            Al[m * SM3_LD + k] = l;
          }
        }
        {
          const int lead = BKC ? kcp : SM_N;
          for (int e = tid; e < SM_N * kcp; e += SM_T) {
            const int q = e / lead, r = e - q * lead;
            const int n = BKC ? q : r, k = BKC ? r : q;
            unsigned short h = 0, l = 0;
            if (n < cols && k < kc) split_bf16(B[tk.b_off + tab[tk.tBK + k0 + k] + tab[tk.tBN + wu.n0 + n]], h, l);
            Bh[n * SM3_LD + k] = h;
            Bl[n * SM3_LD + k] = l;
          }
        }
        __syncthreads();
        const int k8 = 8 * (lane >> 4), ml = 16 * wave + (lane & 15);
        for (int kk = 0; kk < kcp; kk += 32) {
          const bf16x8 ah = *reinterpret_cast<const bf16x8 *>(&Ah[ml * SM3_LD + kk + k8]);
          const bf16x8 al = *reinterpret_cast<const bf16x8 *>(&Al[ml * SM3_LD + kk + k8]);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int nl = 16 * i + (lane & 15);
            const bf16x8 bh = *reinterpret_cast<const bf16x8 *>(&Bh[nl * SM3_LD + kk + k8]);
            const bf16x8 bl = *reinterpret_cast<const bf16x8 *>(&Bl[nl * SM3_LD + kk + k8]);
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, al, acc[i], 0, 0, 0);
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl, ah, acc[i], 0, 0, 0);
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh, ah, acc[i], 0, 0, 0);
          }
        }
      }
    }
    const int ml = 16 * wave + (lane & 15);
    if (wu.slot >= 0) {
      double *P = C + size_t(wu.slot) * (SM_M * SM_N);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) P[(16 * i + 4 * (lane >> 4) + r) * SM_M + ml] = double(acc[i][r]);
      continue;
    }
    const GemmTask t0 = tasks[wu.tbeg];
    const int m = wu.m0 + ml;
    if (m < t0.M) {
      double *Cm = C + t0.c_off + tab[t0.tCM + m];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = wu.n0 + 16 * i + 4 * (lane >> 4) + r;
          if (n < t0.N) {
            double *cp = Cm + tab[t0.tCN + n];
            double v = alpha * double(acc[i][r]);
            if (beta != 0.0) v += beta * (*cp);
            *cp = v;
          }
        }
    }
  }
}

static_assert(SM_T_RED == SM_T, "reduction pass block size");

// Reduction pass of split plans: unit u = {task (for C's tables), first
// slot, m0, n0, end slot}; C tile = alpha * (sum of the slots in order)
// + beta * C.  A is the workspace; deterministic (fixed summation order).
template <int TM, int TN>
__global__ __launch_bounds__(SM_T) void k_reduce_tiles(const double *__restrict__ A,
                                                       const double *__restrict__ B, double *__restrict__ C,
                                                       const GemmTask *__restrict__ tasks,
                                                       const WorkUnit *__restrict__ units, int nunits,
                                                       const int64_t *__restrict__ tab, double alpha,
                                                       double beta) {
  (void)B;
  // one item = one tile x one slice of SM_T of its elements;
  // four independent partial sums keep several loads in flight
  constexpr int PARTS = TM * TN / SM_T;
  for (int w = blockIdx.x; w < nunits * PARTS; w += gridDim.x) {
    const WorkUnit ru = units[w / PARTS];
    const GemmTask t0 = tasks[ru.tbeg];
    const int e = (w % PARTS) * SM_T + threadIdx.x;
    const int n = e / TM, m = e - n * TM;
    if (ru.m0 + m >= t0.M || ru.n0 + n >= t0.N) continue;
    const double *src = A + e;
    double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    int q = ru.tend;
    for (; q + 4 <= ru.slot; q += 4) {
      s0 += src[size_t(q) * (TM * TN)];
      s1 += src[size_t(q + 1) * (TM * TN)];
      s2 += src[size_t(q + 2) * (TM * TN)];
      s3 += src[size_t(q + 3) * (TM * TN)];
    }
    for (; q < ru.slot; ++q) s0 += src[size_t(q) * (TM * TN)];
    const double s = (s0 + s1) + (s2 + s3);
    double *cp = C + t0.c_off + tab[t0.tCM + ru.m0 + m] + tab[t0.tCN + ru.n0 + n];
    double v = alpha * s;
    if (beta != 0.0) v += beta * (*cp);
    *cp = v;
  }
}

// ---- host side --------------------------------------------------------

struct Digit {
  int64_t dim, s1, s2;
};
// A digit set in place (at most ITX_MAX_RANK digits): planning handles one
// per operand side and task, so it must not allocate
struct Digits {
  Digit d[ITX_MAX_RANK];
  int n = 0;
  void push_back(Digit x) { d[n++] = x; }
  bool empty() const { return n == 0; }
  int size() const { return n; }
  const Digit &operator[](int i) const { return d[i]; }
  Digit &back() { return d[n - 1]; }
  const Digit *begin() const { return d; }
  const Digit *end() const { return d + n; }
};

// Remove unit digits and fuse neighbours that are contiguous in both
// operands (the same simplification CProps makes before its GEMM).
void simplify(Digits &d) {
  Digits o;
  for (auto &x : d) {
    if (x.dim == 1) continue;
    if (!o.empty() && o.back().s1 * o.back().dim == x.s1 && o.back().s2 * o.back().dim == x.s2) {
      o.back().dim *= x.dim;
    } else {
      o.push_back(x);
    }
  }
  d = o;
}

int64_t digits_size(const Digits &d) {
  int64_t s = 1;
  for (auto &x : d) s *= x.dim;
  return s;
}

// Offset tables of a plan: every entry is written by ColumnCache::emit, so growing
// the vector leaves new entries uninitialised (default- instead of value-
// initialised: no zeroing pass over the megabytes of a large QN plan).
template <class T>
struct NoInitAlloc : std::allocator<T> {
  template <class U>
  struct rebind {
    using other = NoInitAlloc<U>;
  };
  NoInitAlloc() = default;
  template <class U>
  NoInitAlloc(const NoInitAlloc<U> &) noexcept {}
  template <class U>
  void construct(U *p) noexcept {
    ::new (static_cast<void *>(p)) U;
  }
  template <class U, class... Args>
  void construct(U *p, Args &&...args) {
    ::new (static_cast<void *>(p)) U(std::forward<Args>(args)...);
  }
};
using TabVec = std::vector<int64_t, NoInitAlloc<int64_t>>;

// Offset tables are emitted one column at a time (the A / C row offsets of
// the m digits, B / C of the n digits, A / B of the k digits), each from
// the column's own digit list: the digits with more than one value, merged
// where the column is contiguous by itself (stride of one = dim x stride of
// the previous).  The merged list enumerates the same offsets in the same
// order as the joint digits (first digit fastest) and determines the table,
// so equal columns share one table, and a column that is one run of stride
// 1 (most block rows and k runs) is a prefix of a single 0, 1, 2, ... table.
struct ColDigit {
  int64_t dim, s;
};
int column_digits(const Digits &d, bool first, ColDigit *c) {
  int nc = 0;
  for (auto &x : d) {
    if (x.dim == 1) continue;
    const int64_t st = first ? x.s1 : x.s2;
    if (nc > 0 && c[nc - 1].s * c[nc - 1].dim == st)
      c[nc - 1].dim *= x.dim;
    else
      c[nc++] = ColDigit{x.dim, st};
  }
  return nc;
}

struct ColumnCache {
  struct Key {
    int n;
    ColDigit c[ITX_MAX_RANK];
    bool operator<(const Key &o) const {
      if (n != o.n) return n < o.n;
      for (int i = 0; i < n; ++i) {
        if (c[i].dim != o.c[i].dim) return c[i].dim < o.c[i].dim;
        if (c[i].s != o.c[i].s) return c[i].s < o.c[i].s;
      }
      return false;
    }
  };
  std::map<Key, int64_t> at;
  int64_t iota_start = -1, iota_len = 0;
  // start of the table of column `first` (s1) or not (s2) of d in tab
  int64_t emit(const Digits &d, bool first, TabVec &tab) {
    Key k;
    k.n = column_digits(d, first, k.c);
    int64_t n = 1;
    for (int i = 0; i < k.n; ++i) n *= k.c[i].dim;
    if (n == 0) return int64_t(tab.size());  // an empty extent reads nothing
    if (k.n == 0 || (k.n == 1 && k.c[0].s == 1)) {
      if (iota_len < n) {  // a longer 0, 1, 2, ... table (earlier ones stay valid)
        iota_len = std::max<int64_t>(n, 2 * iota_len);
        iota_start = int64_t(tab.size());
        tab.resize(tab.size() + size_t(iota_len));
        int64_t *t = tab.data() + iota_start;
        for (int64_t x = 0; x < iota_len; ++x) t[x] = x;
      }
      return iota_start;
    }
    auto it = at.find(k);
    if (it != at.end()) return it->second;
    const int64_t start = int64_t(tab.size());
    tab.resize(tab.size() + size_t(n));
    int64_t *t = tab.data() + start;
    // runs along the fastest digit, the other digits advanced once per run
    const int64_t d0 = k.c[0].dim, a0 = k.c[0].s;
    int64_t ctr[ITX_MAX_RANK] = {};
    int64_t o = 0;
    for (int64_t x = 0; x < n; x += d0) {
      for (int64_t i = 0; i < d0; ++i) t[x + i] = o + i * a0;
      for (int i = 1; i < k.n; ++i) {
        ctr[i]++;
        o += k.c[i].s;
        if (ctr[i] < k.c[i].dim) break;
        o -= k.c[i].s * k.c[i].dim;
        ctr[i] = 0;
      }
    }
    at.emplace(k, start);
    return start;
  }
};
// largest offset either table of a digit set holds (strides are positive)
void digits_max(const Digits &d, int64_t &m1, int64_t &m2) {
  m1 = m2 = 0;
  for (auto &x : d) {
    m1 += (x.dim - 1) * x.s1;
    m2 += (x.dim - 1) * x.s2;
  }
}

struct LabelMap {
  // for A index i: contracted partner in B (or -1) / position in C (or -1)
  std::vector<int> a2b, a2c, b2a, b2c;
};

int map_labels(itx_ctx *ctx, int rA, const int32_t *labA, int rB, const int32_t *labB, int rC,
               const int32_t *labC, LabelMap &lm) {
  if (rA < 0 || rB < 0 || rC < 0 || rA > ITX_MAX_RANK || rB > ITX_MAX_RANK || rC > ITX_MAX_RANK)
    return set_err(ctx, ITX_ERR_ARG, "contraction: rank out of range");
  lm.a2b.assign(rA, -1);
  lm.a2c.assign(rA, -1);
  lm.b2a.assign(rB, -1);
  lm.b2c.assign(rB, -1);
  std::vector<int> cused(rC, 0);
  for (int i = 0; i < rA; ++i) {
    if (labA[i] < 0) {
      for (int j = 0; j < rB; ++j)
        if (labB[j] == labA[i]) {
          if (lm.a2b[i] >= 0) return set_err(ctx, ITX_ERR_ARG, "contraction: repeated label in B");
          lm.a2b[i] = j;
          lm.b2a[j] = i;
        }
      if (lm.a2b[i] < 0) return set_err(ctx, ITX_ERR_ARG, "contraction: contracted label of A missing in B");
    } else {
      for (int c = 0; c < rC; ++c)
        if (labC[c] == labA[i]) {
          if (lm.a2c[i] >= 0) return set_err(ctx, ITX_ERR_ARG, "contraction: repeated label in C");
          lm.a2c[i] = c;
          cused[c]++;
        }
      if (lm.a2c[i] < 0) return set_err(ctx, ITX_ERR_ARG, "contraction: label of A missing in C");
    }
  }
  for (int j = 0; j < rB; ++j) {
    if (labB[j] < 0) {
      if (lm.b2a[j] < 0) return set_err(ctx, ITX_ERR_ARG, "contraction: contracted label of B missing in A");
    } else {
      for (int c = 0; c < rC; ++c)
        if (labC[c] == labB[j]) {
          if (lm.b2c[j] >= 0) return set_err(ctx, ITX_ERR_ARG, "contraction: repeated label in C");
          lm.b2c[j] = c;
          cused[c]++;
        }
      if (lm.b2c[j] < 0) return set_err(ctx, ITX_ERR_ARG, "contraction: label of B missing in C");
    }
  }
  for (int c = 0; c < rC; ++c)
    if (cused[c] != 1) return set_err(ctx, ITX_ERR_ARG, "contraction: label of C not found exactly once in A,B");
  return ITX_OK;
}

void colmajor_strides(int r, const int64_t *d, int64_t *s) {
  int64_t x = 1;
  for (int i = 0; i < r; ++i) {
    s[i] = x;
    x *= d[i];
  }
}

// MFMA tiles (BM x BN with GM x GN waves), the skinny and the small-block kernels.
struct TileCfg {
  int bm, bn, gm, gn;
  double eff32;  // relative per-CU efficiency of the reduced forms (MI355X measurements)
};
constexpr TileCfg kTiles[] = {
    {128, 128, 2, 2, 0.70},  // 0
    {128, 64, 2, 2, 1.00},   // 1
    {64, 128, 2, 2, 0.95},   // 2
    {64, 64, 2, 2, 0.95},    // 3
    {32, 32, 2, 2, 0.45},    // 4
    {SK_ROWS, SK_N, 0, 0, 1.0},  // 5: skinny (large M)
    {128, 128, 2, 4, 0.85},  // 6: 8 waves
    {256, 64, 4, 2, 0.55},   // 7: 8 waves
    {64, 256, 2, 4, 1.00},   // 8: 8 waves
    {256, 128, 4, 2, 0.50},  // 9: 8 waves, wave tile 64x64
    {SM_M, SM_N, 0, 0, 1.0},  // 10: small blocks
    {128, 128, 2, 4, 0.85},  // 11: as 6 with 32-deep k stages
    {128, 64, 2, 2, 0.95},   // 12: as 1 with 32-deep k stages
    {64, 128, 2, 2, 0.95},   // 13: as 2 with 32-deep k stages
    {128, 128, 2, 2, 0.85},  // 14: FP32 register-pipelined (k_dgemm); FP64 as 17; k-contiguous pairs only
    {128, 128, 2, 2, 0.85},  // 15: as 14, FP32 two workgroups per CU (k_dgemm2)
    {64, 64, 2, 2, 0.0},     // 16: register-pipelined (k_pipe), FP64 and FP32
    {128, 128, 2, 2, 0.0},   // 17: likewise
    {32, 64, 2, 2, 0.0},     // 18: likewise, FP32
};
constexpr int kNumTiles = 19;
constexpr int kPipe64 = 16, kPipe128 = 17, kPipe32 = 18;
constexpr int kDgemm = 14, kDgemm2 = 15;
constexpr int kSkinny = 5;
static_assert(kSkinny == kSkinnyTile, "tile index of the skinny path");
constexpr int kSmall = 10;
constexpr int kXcds = 8;
constexpr int kSkinnyOcc = 3, kSkinnyQOcc = 4;

// Kernel instantiation of a tile shape, operand layout and form.  All
// kernels of the engine share one argument list (see KernelArgs).
// vec: both operands k-contiguous with aligned runs of 2 (FP64 / FP32
// loaders) or 4 (BF16x3 loader) consecutive k -- the vector-load variants
template <typename T, int BM, int BN, int GM, int GN, int BKS = BK>
const void *gemm_fn(bool akc, bool bkc, bool vec) {
  if (akc && bkc && vec) return reinterpret_cast<const void *>(&k_gemm<T, BM, BN, GM, GN, true, true, BKS, 2>);
  if (akc)
    return bkc ? reinterpret_cast<const void *>(&k_gemm<T, BM, BN, GM, GN, true, true, BKS, 1>)
               : reinterpret_cast<const void *>(&k_gemm<T, BM, BN, GM, GN, true, false, BKS, 1>);
  return bkc ? reinterpret_cast<const void *>(&k_gemm<T, BM, BN, GM, GN, false, true, BKS, 1>)
             : reinterpret_cast<const void *>(&k_gemm<T, BM, BN, GM, GN, false, false, BKS, 1>);
}

template <int BM, int BN, int GM, int GN>
const void *gemm3_fn(bool akc, bool bkc, bool vec, bool split = false) {
  if (split)  // pre-split operands: k-contiguous layouts only
    return vec ? reinterpret_cast<const void *>(&k_gemm3<BM, BN, GM, GN, true, true, 4, true>)
               : reinterpret_cast<const void *>(&k_gemm3<BM, BN, GM, GN, true, true, 1, true>);
  if (akc && bkc && vec) return reinterpret_cast<const void *>(&k_gemm3<BM, BN, GM, GN, true, true, 4>);
  if (akc)
    return bkc ? reinterpret_cast<const void *>(&k_gemm3<BM, BN, GM, GN, true, true, 1>)
               : reinterpret_cast<const void *>(&k_gemm3<BM, BN, GM, GN, true, false, 1>);
  return bkc ? reinterpret_cast<const void *>(&k_gemm3<BM, BN, GM, GN, false, true, 1>)
             : reinterpret_cast<const void *>(&k_gemm3<BM, BN, GM, GN, false, false, 1>);
}

template <typename T, int FM, int FN>
const void *pipe_fn(bool akc, bool bkc, bool vec, bool split = false) {
  constexpr int V = sizeof(T) == 2 ? 4 : 2;
  if constexpr (sizeof(T) == 2) {
    if (split)
      return vec ? reinterpret_cast<const void *>(&k_pipe<T, FM, FN, V, V, true>)
                 : reinterpret_cast<const void *>(&k_pipe<T, FM, FN, 1, 1, true>);
  }
  if (akc && bkc && vec) return reinterpret_cast<const void *>(&k_pipe<T, FM, FN, V, V>);
  if (akc)
    return bkc ? reinterpret_cast<const void *>(&k_pipe<T, FM, FN, 1, 1>)
               : reinterpret_cast<const void *>(&k_pipe<T, FM, FN, 1, 0>);
  return bkc ? reinterpret_cast<const void *>(&k_pipe<T, FM, FN, 0, 1>)
             : reinterpret_cast<const void *>(&k_pipe<T, FM, FN, 0, 0>);
}

const void *gemm3_fn_tile(int tile, bool akc, bool bkc, bool vec, bool split) {
  switch (tile) {
    case 0: return gemm3_fn<128, 128, 2, 2>(akc, bkc, vec, split);
    case 1: return gemm3_fn<128, 64, 2, 2>(akc, bkc, vec, split);
    case 2: return gemm3_fn<64, 128, 2, 2>(akc, bkc, vec, split);
    case 3: return gemm3_fn<64, 64, 2, 2>(akc, bkc, vec, split);
    case 6: return gemm3_fn<128, 128, 2, 4>(akc, bkc, vec, split);
    case 7: return gemm3_fn<256, 64, 4, 2>(akc, bkc, vec, split);
    case 8: return gemm3_fn<64, 256, 2, 4>(akc, bkc, vec, split);
    case 9: return gemm3_fn<256, 128, 4, 2>(akc, bkc, vec, split);
    case 11: return gemm3_fn<128, 128, 2, 4>(akc, bkc, vec, split);
    case 12: return gemm3_fn<128, 64, 2, 2>(akc, bkc, vec, split);
    case 13: return gemm3_fn<64, 128, 2, 2>(akc, bkc, vec, split);
    case 14:
    case 15: return gemm3_fn<128, 128, 2, 2>(akc, bkc, vec, split);  // not chosen for BF16x3
    case 16: return pipe_fn<unsigned short, 2, 2>(akc, bkc, vec, split);
    case 17: return pipe_fn<unsigned short, 4, 4>(akc, bkc, vec, split);
    default: return gemm3_fn<32, 32, 2, 2>(akc, bkc, vec, split);
  }
}

template <typename T>
const void *gemm_fn_tile(int tile, bool akc, bool bkc, bool vec) {
  switch (tile) {
    case 0: return gemm_fn<T, 128, 128, 2, 2>(akc, bkc, vec);
    case 1: return gemm_fn<T, 128, 64, 2, 2>(akc, bkc, vec);
    case 2: return gemm_fn<T, 64, 128, 2, 2>(akc, bkc, vec);
    case 3: return gemm_fn<T, 64, 64, 2, 2>(akc, bkc, vec);
    case 6: return gemm_fn<T, 128, 128, 2, 4>(akc, bkc, vec);
    case 7: return gemm_fn<T, 256, 64, 4, 2>(akc, bkc, vec);
    case 8: return gemm_fn<T, 64, 256, 2, 4>(akc, bkc, vec);
    case 9: return gemm_fn<T, 256, 128, 4, 2>(akc, bkc, vec);
    case 11: return gemm_fn<T, 128, 128, 2, 4, 32>(akc, bkc, vec);
    case 12: return gemm_fn<T, 128, 64, 2, 2, 32>(akc, bkc, vec);
    case 13: return gemm_fn<T, 64, 128, 2, 2, 32>(akc, bkc, vec);
    case 14:  // k-contiguous operands in aligned pairs; otherwise FP32 tile 0's kernel
    case 15:
      if constexpr (std::is_same_v<T, double>) {
        return pipe_fn<T, 4, 4>(akc, bkc, vec);
      } else {
        if (akc && bkc && vec)
          return tile == 14 ? reinterpret_cast<const void *>(&k_dgemm<T>) : reinterpret_cast<const void *>(&k_dgemm2<T>);
        return gemm_fn<T, 128, 128, 2, 2>(akc, bkc, false);
      }
    case 16: return pipe_fn<T, 2, 2>(akc, bkc, vec);
    case 17: return pipe_fn<T, 4, 4>(akc, bkc, vec);
    case 18:  // FP32 only (build_plan)
      if constexpr (std::is_same_v<T, float>) return pipe_fn<T, 1, 2>(akc, bkc, vec);
      return nullptr;
    default: return gemm_fn<T, 32, 32, 2, 2>(akc, bkc, vec);
  }
}

// What the skinny path's variants depend on.
struct Skinny {
  int maxn = SK_N;    // largest N of the tasks
  bool tiny = false;  // every task has K <= 8 and N <= 8
  int slots = 0;      // of 4 k, one task per C block (0: several, or K > 4 SK_KS)
};

template <int NB>
const void *skinny_fn(int slots) {
  return slots == 0   ? reinterpret_cast<const void *>(&k_skinny<NB, 0>)
         : slots == 1 ? reinterpret_cast<const void *>(&k_skinny<NB, 1>)
         : slots <= 3 ? reinterpret_cast<const void *>(&k_skinny<NB, 3>)
                      : reinterpret_cast<const void *>(&k_skinny<NB, SK_KS>);
}

// Entry point and workgroup size of a plan's kernel.
const void *kernel_of(int tile, int prec, bool akc, bool bkc, int *block, int vec = 0, bool split = false,
                      Skinny sk = Skinny{}) {
  if (tile == kSkinny) {  // HBM-bound: FP64 arithmetic in every form
    *block = SK_ROWS;
    if (sk.tiny) return reinterpret_cast<const void *>(&k_skinny_q);
    return sk.maxn <= 16 ? skinny_fn<1>(sk.slots) : skinny_fn<2>(sk.slots);
  }
  if (tile == kSmall) {
    *block = SM_T;
    if (prec == ITX_PREC_F32) {
      if (akc) return bkc ? reinterpret_cast<const void *>(&k_small_f32<true, true>)
                          : reinterpret_cast<const void *>(&k_small_f32<true, false>);
      return bkc ? reinterpret_cast<const void *>(&k_small_f32<false, true>)
                 : reinterpret_cast<const void *>(&k_small_f32<false, false>);
    }
    if (prec == ITX_PREC_BF16X3) {
      if (akc) return bkc ? reinterpret_cast<const void *>(&k_small_bf16x3<true, true>)
                          : reinterpret_cast<const void *>(&k_small_bf16x3<true, false>);
      return bkc ? reinterpret_cast<const void *>(&k_small_bf16x3<false, true>)
                 : reinterpret_cast<const void *>(&k_small_bf16x3<false, false>);
    }
    *block = SMD_T;
    if (akc) return bkc ? reinterpret_cast<const void *>(&k_small<true, true>)
                        : reinterpret_cast<const void *>(&k_small<true, false>);
    return bkc ? reinterpret_cast<const void *>(&k_small<false, true>)
               : reinterpret_cast<const void *>(&k_small<false, false>);
  }
  *block = 64 * kTiles[tile].gm * kTiles[tile].gn;
  // vec: bit 0 = runs of 2 usable (FP64 / FP32), bit 1 = runs of 4 (BF16x3),
  // bit 2 = runs of 4 on 4-element boundaries (BF16x3 pre-split words)
  if (prec == ITX_PREC_BF16X3)
    return gemm3_fn_tile(tile, akc, bkc, split ? (vec & 4) != 0 : (vec & 2) != 0, split);
  return prec == ITX_PREC_F64 ? gemm_fn_tile<double>(tile, akc, bkc, (vec & 1) != 0)
                              : gemm_fn_tile<float>(tile, akc, bkc, (vec & 1) != 0);
}

// Resident workgroups per CU of one kernel instantiation (registers and
// LDS), from the runtime's occupancy calculator; cached per variant.
int tile_occupancy(int tile, int prec, bool akc, bool bkc) {
  static std::map<int, int> cache;
  if (tile == kSkinny) return kSkinnyOcc;
  const int key = tile * 16 + prec * 4 + (akc ? 2 : 0) + (bkc ? 1 : 0);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  int block = 0, nb = 0;
  const void *f = kernel_of(tile, prec, akc, bkc, &block, (tile == kDgemm || tile == kDgemm2) ? 1 : 0);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, block, 0) != hipSuccess || nb < 1) {
    (void)hipGetLastError();
    nb = 1;
  }
  cache[key] = nb;
  return nb;
}

// lpt_makespan of n units of one cost
double lpt_makespan(int64_t n, double cost, int64_t slots) {
  if (n > 4 * slots) return double(n) * cost / double(slots) + 0.5 * cost;
  return double((n + slots - 1) / slots) * cost;
}

// Makespan of units (costs) on `slots` identical workers, heaviest first
// onto the least loaded worker (what the persistent loop approximates).
double lpt_makespan(std::vector<double> costs, int64_t slots) {
  if (costs.empty()) return 0;
  if (int64_t(costs.size()) <= slots) return *std::max_element(costs.begin(), costs.end());
  if (int64_t(costs.size()) > 4 * slots) {
    // many more units than slots: LPT ends within one unit of the load
    // bound, which is what the comparison between tiles needs
    double sum = 0, mx = 0;
    for (double c : costs) {
      sum += c;
      mx = std::max(mx, c);
    }
    return std::max(mx, sum / double(slots) + 0.5 * mx);
  }
  std::sort(costs.begin(), costs.end(), std::greater<double>());
  std::priority_queue<double, std::vector<double>, std::greater<double>> q;
  for (int64_t i = 0; i < slots; ++i) q.push(0.0);
  double mk = 0;
  for (double c : costs) {
    double t = q.top() + c;
    q.pop();
    q.push(t);
    mk = std::max(mk, t);
  }
  return mk;
}

// Size class of a contraction for the tuning table: precision, operand
// contiguity, and log2 buckets of the largest C block, summed K, #blocks.
std::string tune_key(int prec, bool akc, bool bkc, int maxM, int maxN, double maxKsum, int ngroups) {
  auto lg = [](double x) { return int(std::ceil(std::log2(std::max(1.0, x)))); };
  char b[96];
  std::snprintf(b, sizeof b, "p%d a%d b%d M%d N%d K%d G%d", prec, int(akc), int(bkc), lg(maxM), lg(maxN),
                lg(maxKsum), lg(ngroups));
  return b;
}

}  // namespace

int build_plan(itx_ctx *ctx, int rA, const int32_t *labA, int rB, const int32_t *labB, int rC,
               const int32_t *labC, int ntasks, const int64_t *offs, const int64_t *blkA,
               const int64_t *blkB, const int64_t *blkC, int prec, itx_plan **out, void *into,
               size_t into_cap) {
  *out = nullptr;
  if (prec != ITX_PREC_F64 && prec != ITX_PREC_F32 && prec != ITX_PREC_BF16X3)
    return set_err(ctx, ITX_ERR_ARG, "contraction: unknown precision form");
  if (ntasks < 0) return set_err(ctx, ITX_ERR_ARG, "contraction: negative task count");
  LabelMap lm;
  int rc = map_labels(ctx, rA, labA, rB, labB, rC, labC, lm);
  if (rc) return rc;

  std::vector<GemmTask> tasks;
  TabVec tab;
  ColumnCache ccache;
  tasks.reserve(ntasks);
  // operand extents (elements) for the autotuner's scratch buffers
  int64_t extA = 1, extB = 1, extC = 1;
  // A is read along k if its unit-stride digit is a contracted one (else
  // along m); likewise B.  Decided on the first non-empty task.
  bool first_kc = false;  // of the first task
  double akc_work = 0, bkc_work = 0;  // multiply-adds of tasks with k-contiguous operands less those of the others
  double run_work = 0;                // those of tasks with no operand in short runs, less those of the others

  double flops = 0;
  // Everything a task needs besides its offsets follows from the block
  // dims of its A and B blocks; QN task lists repeat few distinct dims, so
  // the analysis (GEMM digits, offset tables, extents) is done once per
  // distinct (dims A, dims B) and looked up for the other tasks.
  struct DimInfo {
    int64_t dC[ITX_MAX_RANK];
    int32_t M, N, K;
    int64_t tAM, tCM, tBN, tCN, tAK, tBK;
    int64_t am, cm, bn, cn, ak, bk;
    bool akc, bkc, empty;
    bool arow, brow;  // read along the rows (columns of B), in runs of 16 or all
    int vec;  // bit 0: k runs of 2 usable by both operands, bit 1: runs of 4 (bit 2: below)
  };
  std::vector<DimInfo> infos;
  std::vector<int64_t> ikeys;  // the dims of each entry (rA + rB per entry)
  std::unordered_map<uint64_t, int> icache;
  const int rAB = rA + rB;
  auto analyze = [&](const int64_t *dA, const int64_t *dB, DimInfo &fi) -> int {
    int64_t sA[ITX_MAX_RANK], sB[ITX_MAX_RANK], sC[ITX_MAX_RANK];
    int64_t *dC = fi.dC;
    for (int i = 0; i < rA; ++i) {
      if (dA[i] < 0) return set_err(ctx, ITX_ERR_ARG, "contraction: negative dimension");
      if (lm.a2b[i] >= 0 && dB[lm.a2b[i]] != dA[i])
        return set_err(ctx, ITX_ERR_ARG, "contraction: contracted dimensions differ");
      if (lm.a2c[i] >= 0) dC[lm.a2c[i]] = dA[i];
    }
    for (int j = 0; j < rB; ++j) {
      if (dB[j] < 0) return set_err(ctx, ITX_ERR_ARG, "contraction: negative dimension");
      if (lm.b2c[j] >= 0) dC[lm.b2c[j]] = dB[j];
    }
    colmajor_strides(rA, dA, sA);
    colmajor_strides(rB, dB, sB);
    colmajor_strides(rC, dC, sC);
    Digits dm, dn, dk;
    for (int i = 0; i < rA; ++i) {
      if (lm.a2c[i] >= 0) dm.push_back({dA[i], sA[i], sC[lm.a2c[i]]});
      else dk.push_back({dA[i], sA[i], sB[lm.a2b[i]]});
    }
    for (int j = 0; j < rB; ++j)
      if (lm.b2c[j] >= 0) dn.push_back({dB[j], sB[j], sC[lm.b2c[j]]});
    simplify(dm);
    simplify(dn);
    simplify(dk);
    const int64_t M = digits_size(dm), N = digits_size(dn), K = digits_size(dk);
    if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX)
      return set_err(ctx, ITX_ERR_UNSUPPORTED, "contraction: GEMM extent exceeds 2^31");
    fi.M = int32_t(M);
    fi.N = int32_t(N);
    fi.K = int32_t(K);
    fi.empty = (M == 0 || N == 0);  // empty C block: nothing to write
    if (fi.empty) return ITX_OK;
    {
      int64_t na = 1, nb = 1, nc = 1;
      for (int i = 0; i < rA; ++i) na *= dA[i];
      for (int j = 0; j < rB; ++j) nb *= dB[j];
      for (int c = 0; c < rC; ++c) nc *= dC[c];
      if (na > INT32_MAX || nb > INT32_MAX || nc > INT32_MAX)
        return set_err(ctx, ITX_ERR_UNSUPPORTED, "contraction: a block of 2^31 or more elements");
    }
    fi.akc = !dk.empty() && dk[0].s1 == 1;
    fi.bkc = !dk.empty() && dk[0].s2 == 1;
    fi.tAM = ccache.emit(dm, true, tab);
    fi.tCM = ccache.emit(dm, false, tab);
    fi.tBN = ccache.emit(dn, true, tab);
    fi.tCN = ccache.emit(dn, false, tab);
    fi.tAK = ccache.emit(dk, true, tab);
    fi.tBK = ccache.emit(dk, false, tab);
    digits_max(dm, fi.am, fi.cm);
    digits_max(dn, fi.bn, fi.cn);
    digits_max(dk, fi.ak, fi.bk);
    // vector loads: both operands k-contiguous, every aligned group of V
    // consecutive k one run of V consecutive elements starting at an even
    // offset, every row offset even (16-byte aligned given an aligned base)
    fi.vec = 0;
    // Decided from the digits instead of scanning the tables: one column of
    // a digit set (s1 or s2) re-merged where it is contiguous by itself;
    // every offset of that table is a multiple of `al` iff every stride is,
    // and the table comes in runs of V consecutive offsets starting at
    // multiples of `al` iff V divides its size, the fastest digit has
    // stride 1 and a multiple of V entries, and the other strides are
    // multiples of `al` (checked against the table scan on random digit
    // sets, both columns, V = 2, 4 and al = 2, 4)
    auto column = [](const Digits &d, bool first, Digit *c) {
      int nc = 0;
      for (auto &x : d) {
        if (x.dim == 1) continue;
        const int64_t st = first ? x.s1 : x.s2;
        if (nc > 0 && c[nc - 1].s1 * c[nc - 1].dim == st)
          c[nc - 1].dim *= x.dim;
        else
          c[nc++] = Digit{x.dim, st, 0};
      }
      return nc;
    };
    auto aligned = [&](const Digits &d, bool first, int al) {
      Digit c[ITX_MAX_RANK];
      const int nc = column(d, first, c);
      for (int i = 0; i < nc; ++i)
        if (c[i].s1 % al) return false;
      return true;
    };
    auto runs = [&](const Digits &d, bool first, int64_t n, int V, int al) {
      if (n % V) return false;
      Digit c[ITX_MAX_RANK];
      const int nc = column(d, first, c);
      if (nc == 0 || c[0].s1 != 1 || c[0].dim % V) return false;
      for (int i = 1; i < nc; ++i)
        if (c[i].s1 % al) return false;
      return true;
    };
    auto row_runs = [&](const Digits &d, int64_t n) {
      Digit c[ITX_MAX_RANK];
      return column(d, true, c) > 0 && c[0].s1 == 1 && c[0].dim >= std::min<int64_t>(16, n);
    };
    fi.arow = !fi.akc && row_runs(dm, M);
    fi.brow = !fi.bkc && row_runs(dn, N);
    if (fi.akc && fi.bkc) {
      if (aligned(dm, true, 2) && aligned(dn, true, 2)) {
        if (runs(dk, true, K, 2, 2) && runs(dk, false, K, 2, 2)) fi.vec |= 1;
        if (runs(dk, true, K, 4, 2) && runs(dk, false, K, 4, 2)) fi.vec |= 2;
      }
      if (aligned(dm, true, 4) && aligned(dn, true, 4) && runs(dk, true, K, 4, 4) && runs(dk, false, K, 4, 4))
        fi.vec |= 4;
    }
    return ITX_OK;
  };
  int vecbits = 7;  // AND over the tasks
  for (int t = 0; t < ntasks; ++t) {
    const int64_t *dA = blkA + size_t(t) * rA;
    const int64_t *dB = blkB + size_t(t) * rB;
    uint64_t h = 1469598103934665603ull;  // FNV-1a over the dims
    for (int i = 0; i < rA; ++i) h = (h ^ uint64_t(dA[i])) * 1099511628211ull;
    for (int j = 0; j < rB; ++j) h = (h ^ uint64_t(dB[j])) * 1099511628211ull;
    const DimInfo *fp = nullptr;
    auto it = icache.find(h);
    if (it != icache.end()) {
      const int64_t *kd = ikeys.data() + size_t(it->second) * rAB;
      if (std::equal(dA, dA + rA, kd) && std::equal(dB, dB + rB, kd + rA)) fp = &infos[size_t(it->second)];
    }
    DimInfo tmp;
    if (!fp) {
      int rc2 = analyze(dA, dB, tmp);
      if (rc2) return rc2;
      if (it == icache.end()) {  // first dims with this hash: remember them
        icache.emplace(h, int(infos.size()));
        ikeys.insert(ikeys.end(), dA, dA + rA);
        ikeys.insert(ikeys.end(), dB, dB + rB);
        infos.push_back(tmp);
        fp = &infos.back();
      } else {
        fp = &tmp;
      }
    }
    const DimInfo &fi = *fp;
    if (blkC) {
      for (int c = 0; c < rC; ++c)
        if (blkC[size_t(t) * rC + c] != fi.dC[c])
          return set_err(ctx, ITX_ERR_ARG, "contraction: dimensions of C do not match A and B");
    }
    if (fi.empty) continue;
    // the tasks' common layout, by their work (K = 1 has none: at chi = 750
    // the first block of the chain's products is 1 x 1 x 1)
    if (tasks.empty()) first_kc = fi.akc && fi.bkc;
    const double work = fi.K > 1 ? double(fi.M) * double(fi.N) * double(fi.K) : 0.0;
    akc_work += fi.akc ? work : -work;
    bkc_work += fi.bkc ? work : -work;
    run_work += (fi.akc || fi.arow) && (fi.bkc || fi.brow) ? work : -work;
    vecbits &= fi.vec;
    if (offs[3 * size_t(t)] % 2 || offs[3 * size_t(t) + 1] % 2) vecbits = 0;
    if (offs[3 * size_t(t)] % 4 || offs[3 * size_t(t) + 1] % 4) vecbits &= ~4;
    GemmTask g{};
    g.a_off = offs[3 * size_t(t)];
    g.b_off = offs[3 * size_t(t) + 1];
    g.c_off = offs[3 * size_t(t) + 2];
    g.M = fi.M;
    g.N = fi.N;
    g.K = fi.K;
    g.tAM = fi.tAM;
    g.tCM = fi.tCM;
    g.tBN = fi.tBN;
    g.tCN = fi.tCN;
    g.tAK = fi.tAK;
    g.tBK = fi.tBK;
    extA = std::max(extA, g.a_off + fi.am + fi.ak + 1);
    extB = std::max(extB, g.b_off + fi.bk + fi.bn + 1);
    extC = std::max(extC, g.c_off + fi.cm + fi.cn + 1);
    flops += 2.0 * double(fi.M) * double(fi.N) * double(fi.K);
    tasks.push_back(g);
  }
  const bool akc = akc_work > 0, bkc = bkc_work > 0;

  // group tasks by C block, in C offset order and stable within a block
  // (keeps the planner's pair order): a counting sort over the distinct
  // C offsets
  std::vector<GemmTask> st(tasks.size());
  {
    // C offset -> bucket (first-appearance numbering) through an
    // open-addressing table, then buckets renumbered in offset order
    size_t cap = 16;
    while (cap < 2 * tasks.size()) cap <<= 1;
    std::vector<int64_t> hk(cap, -1);
    std::vector<int> hv(cap, 0), bucket(tasks.size());
    std::vector<int64_t> first;  // distinct C offsets, first-appearance order
    for (size_t i = 0; i < tasks.size(); ++i) {
      const int64_t c = tasks[i].c_off;
      size_t h = size_t((uint64_t(c) * 0x9E3779B97F4A7C15ull) >> 20) & (cap - 1);
      while (hk[h] != -1 && hk[h] != c) h = (h + 1) & (cap - 1);
      if (hk[h] == -1) {
        hk[h] = c;
        hv[h] = int(first.size());
        first.push_back(c);
      }
      bucket[i] = hv[h];
    }
    std::vector<int> ord(first.size()), rank(first.size());
    std::iota(ord.begin(), ord.end(), 0);
    std::sort(ord.begin(), ord.end(), [&](int x, int y) { return first[size_t(x)] < first[size_t(y)]; });
    for (size_t r = 0; r < ord.size(); ++r) rank[size_t(ord[r])] = int(r);
    std::vector<int> cnt(first.size() + 1, 0);
    for (size_t i = 0; i < tasks.size(); ++i) {
      bucket[i] = rank[size_t(bucket[i])];
      ++cnt[size_t(bucket[i]) + 1];
    }
    for (size_t b = 1; b < cnt.size(); ++b) cnt[b] += cnt[b - 1];
    for (size_t i = 0; i < tasks.size(); ++i) st[size_t(cnt[size_t(bucket[i])]++)] = tasks[i];
  }
  struct Grp {
    int tb, te;
    int M, N;
    double ksum;
  };
  std::vector<Grp> groups;
  for (size_t i = 0; i < st.size();) {
    size_t e = i + 1;
    while (e < st.size() && st[e].c_off == st[i].c_off) {
      if (st[e].M != st[i].M || st[e].N != st[i].N)
        return set_err(ctx, ITX_ERR_ARG, "contraction: tasks writing one C block disagree on its shape");
      ++e;
    }
    double ks = 0;
    for (size_t q = i; q < e; ++q) ks += st[q].K;
    groups.push_back({int(i), int(e), st[i].M, st[i].N, ks});
    i = e;
  }

  const int cus = std::max(1, ctx->num_cus);
  int maxN = 0, maxK = 0, maxM = 0;
  double maxKsum = 0;
  for (auto &t : st) {
    maxN = std::max(maxN, t.N);
    maxK = std::max(maxK, t.K);
    maxM = std::max(maxM, t.M);
  }
  for (auto &g : groups) maxKsum = std::max(maxKsum, g.ksum);

  // Build the device plan for one tile choice.
  // tiles 14 and 15 need k-contiguous operands in aligned pairs
  const bool dg_ok = (prec == ITX_PREC_F64 || prec == ITX_PREC_F32) && akc && bkc && (vecbits & 1);
  auto tile_ok = [&](int t) {
    return ((t != kDgemm && t != kDgemm2) || dg_ok) && (t != kPipe32 || prec == ITX_PREC_F32);
  };
  // skinny plans whose tasks all have K, N <= 8 run k_skinny_q: two rows per thread
  const bool tinyq = maxN <= SKQ_N && maxK <= SKQ_K;
  bool lean = false;  // a caller's scratch is too small for more and finer units
  // Units over k of the 64 x 64 tile for one product: as many as give every
  // CU two workgroups, with at least 8 stages each.
  auto pipe_split = [&]() {
    if (st.size() != 1 || lean || prec != ITX_PREC_F64) return 1;  // FP32 sums keep their order
    const int64_t tiles = int64_t((st[0].M + 63) / 64) * ((st[0].N + 63) / 64);
    const int64_t most = std::min<int64_t>(2 * cus / std::max<int64_t>(tiles, 1), st[0].K / (8 * DG_BK));
    return int(std::max<int64_t>(1, std::min<int64_t>(most, 64)));
  };
  auto finalize = [&](int best, itx_plan **pout) -> int {
    *pout = nullptr;
    if (!tile_ok(best)) return ITX_ERR_UNSUPPORTED;
    const int tbm0 = (best == kSkinny && tinyq) ? SKQ_R * SK_ROWS : kTiles[best].bm;
    const int tbn0 = (best == kSkinny) ? std::max(1, maxN) : kTiles[best].bn;
    int tbm = tbm0, tbn = tbn0;
    if (best == kSmall && prec == ITX_PREC_F64 && !lean) {
      // Smaller units while they leave CUs idle: a unit's k loop is bound by
      // the matrix cores of one CU (64 x 32 outputs: 32 cycles a k), its loads
      // by its rows, so two units of half the size take half the time.  One
      // 128 x 32 block with K = 160: 9.2 us as two units, 5 us as 16.
      auto count = [&](int bm, int bn) {
        int64_t n = 0;
        for (auto &g : groups) n += int64_t((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn);
        return n;
      };
      if (count(64, 32) < cus) tbm = 32;
      if (count(32, 32) < cus / 2) tbm = tbn = 16;
    }
    std::vector<WorkUnit> units, red;
    std::vector<double> ucost;
    std::vector<GemmTask> vt;  // device task list (st, or its k-chunks when split)
    int nslots = 0;
    bool split = false;
    const int slot_elems = best == kPipe64 ? 64 * 64 : SM_M * SM_N;
    if (const int ns = best == kPipe64 ? pipe_split() : 1; ns > 1) {
      // The k of a product with few tiles over several units: the k ranges
      // outermost, so that an XCD's units share one range of A and B.
      split = true;
      const Grp &g = groups[0];
      const int kc = ((st[0].K + ns - 1) / ns + DG_BK - 1) / DG_BK * DG_BK;
      std::vector<std::array<int, 2>> at;
      for (int m0 = 0; m0 < g.M; m0 += 64)
        for (int n0 = 0; n0 < g.N; n0 += 64) at.push_back({m0, n0});
      const int nk = (st[0].K + kc - 1) / kc;
      for (int i = 0; i < nk; ++i) {
        GemmTask x = st[0];
        x.K = std::min(kc, st[0].K - i * kc);
        x.tAK += i * kc;
        x.tBK += i * kc;
        vt.push_back(x);
        for (size_t j = 0; j < at.size(); ++j) {
          units.push_back({i, i + 1, at[j][0], at[j][1], int(j) * nk + i, 0});
          ucost.push_back(0.0);  // in this order
        }
      }
      for (size_t j = 0; j < at.size(); ++j) red.push_back({0, int(j) * nk, at[j][0], at[j][1], int(j + 1) * nk, 0});
      nslots = int(at.size()) * nk;
    } else if (best == kSmall) {
      // Split the k-chunk sequence of heavy tiles over several units when
      // the tiles alone cannot fill the device (few C blocks, long task
      // lists): chunk budget c per unit from the total work.
      double total = 0, maxw = 0;
      for (auto &g : groups) {
        double w = 0;
        for (int t = g.tb; t < g.te; ++t) w += double((st[t].K + SM_K - 1) / SM_K);
        const double tiles = double((g.M + tbm0 - 1) / tbm0) * double((g.N + tbn0 - 1) / tbn0);
        total += w * tiles;
        maxw = std::max(maxw, w);
      }
      const double target = 2.0 * cus * tile_occupancy(kSmall, prec, akc, bkc);
      const double c = std::max(1.0, std::ceil(total / target));
      // Units of at least `least` k-chunks: reduced forms two (a one-chunk unit
      // writes a partial tile for as many bytes as it reads); FP64 eight, one
      // for each wave of a unit, which share its chunks anyway -- a split
      // costs a second launch (4 us) where a chunk more costs a trip to memory
      const int least = prec == ITX_PREC_F64 ? SMD_W : 2;
      split = maxw > 2.0 * std::max(c, prec == ITX_PREC_F64 ? double(least) : 1.0) && total * (SM_M * SM_N) * 8.0 / c < double(size_t(1) << 30);
      if (split) {
        tbm = tbm0;  // partial tiles are whole
        tbn = tbn0;
        const int per = std::max(least, int(c));
        for (auto &g : groups) {
          const int vb = int(vt.size());
          for (int t = g.tb; t < g.te; ++t)
            for (int k0 = 0; k0 < st[t].K; k0 += SM_K) {
              GemmTask x = st[t];
              x.K = std::min(SM_K, st[t].K - k0);
              x.tAK += k0;
              x.tBK += k0;
              vt.push_back(x);
            }
          const int ve = int(vt.size());
          for (int m0 = 0; m0 < g.M; m0 += tbm)
            for (int n0 = 0; n0 < g.N; n0 += tbn) {
              const int s0 = nslots;
              for (int a = vb; a < ve; a += per) {
                units.push_back({a, std::min(ve, a + per), m0, n0, nslots++, tbm | tbn << 8});
                ucost.push_back(double(std::min(ve, a + per) - a));
              }
              red.push_back({vb, s0, m0, n0, nslots, 0});
            }
        }
      }
    }
    if (!split) {
      vt = st;
      // Tiles of a C block in super-tiles of SUPM x SUPN: the 32 workgroups
      // an XCD runs side by side then share 4 row blocks of A and 8 column
      // blocks of B in that XCD's L2 (m-major order shares one row block
      // with 32 column blocks, re-reading B once per row block).
      const int SUPM = 4, SUPN = 8;
      for (auto &g : groups) {
        const int tm = (g.M + tbm - 1) / tbm, tn = (g.N + tbn - 1) / tbn;
        for (int sm = 0; sm < tm; sm += SUPM)
          for (int sn = 0; sn < tn; sn += SUPN)
            for (int im = sm; im < std::min(tm, sm + SUPM); ++im)
              for (int in = sn; in < std::min(tn, sn + SUPN); ++in) {
                units.push_back({g.tb, g.te, im * tbm, in * tbn, -1, best == kSmall ? tbm | tbn << 8 : 0});
                ucost.push_back(g.ksum);
              }
      }
    }
    // heaviest units first (the persistent loop then balances like LPT);
    // stable so equal-cost tiles keep their m-major order
    {
      std::vector<std::pair<double, int>> ui(units.size());
      bool sorted = true;
      for (size_t i = 0; i < units.size(); ++i) {
        ui[i] = {-ucost[i], int(i)};  // (cost descending, position ascending): the stable order
        sorted = sorted && (i == 0 || ucost[i] <= ucost[i - 1]);
      }
      if (!sorted) {
        std::sort(ui.begin(), ui.end());
        std::vector<WorkUnit> su(units.size());
        for (size_t i = 0; i < ui.size(); ++i) {
          su[i] = units[size_t(ui[i].second)];
          ucost[i] = -ui[i].first;
        }
        units.swap(su);
      }
    }
    if (groups.size() > 1 && !split ? units.size() > size_t(cus)
                                    : best != kSkinny && units.size() > 2 * kXcds &&
                                          (groups.size() > 1 || !split || best == kPipe64)) {
      // Workgroup b runs on XCD b % 8 and takes units b, b + grid, ...: each
      // XCD gets a list of units that share operands in its L2.  Equal units
      // (one block, or the pieces of a product split over k): eighths of the list.  Several
      // blocks: pieces of at most 1/24 of the work spread by their cost, a
      // piece the tiles of one block (they share rows of A and columns of B)
      // or, for narrow tasks, the tiles at the same rows of the blocks that
      // read the same blocks of A (B is a few numbers; an MPO stage reads
      // each block of A for every channel it feeds).  chi = 1024 block-sparse
      // chain, against the blocks from the heaviest down: 29.5 to 23.6, 23.4
      // to 19.3 and 38.6 to 28.4 us; up to a unit per CU it gains nothing.  The
      // pieces of one split small block stay in their order, a tile's k ranges
      // round robin: its tiles then meet the same k on an XCD (90 x 90 x 60000 in
      // FP32 150 us as eighths, 125 in order); those of several blocks, whose
      // tiles share less, do not (chain at chi = 640, last stage in BF16x3 25 us as
      // eighths, 32 in order).
      const size_t n = units.size();
      std::vector<WorkUnit> su;
      su.reserve(n);
      if (split || groups.size() == 1) {
        // the first n % 8 XCDs have one more: every round of eight is whole
        const size_t len = n / kXcds, more = n % kXcds;
        for (size_t i = 0; i < n; ++i) {
          const size_t x = i % kXcds;
          su.push_back(units[x * len + std::min(x, more) + i / kXcds]);
        }
      } else {
        std::array<std::vector<WorkUnit>, kXcds> lists;
        std::vector<int> head(vt.size());  // a block's first task -> its place in `open`
        std::iota(head.begin(), head.end(), 0);
        std::vector<int> open(vt.size(), -1);  // the latest piece of a block, or of a set's tile of rows
        if (best == kSkinny) {
          auto root = [&](int t) {
            while (head[size_t(t)] != t) t = head[size_t(t)] = head[size_t(head[size_t(t)])];
            return t;
          };
          std::unordered_map<int64_t, int> reader(2 * vt.size());  // block of A -> a block that reads it
          for (auto &g : groups)
            for (int t = g.tb; t < g.te; ++t)
              head[size_t(root(g.tb))] = root(reader.emplace(vt[size_t(t)].a_off, g.tb).first->second);
          std::vector<int> rows(vt.size(), 0);  // of a set, in tiles; then its place in `open`
          for (auto &g : groups) {
            int &r = rows[size_t(root(g.tb))];
            r = std::max(r, (g.M + tbm - 1) / tbm);
          }
          int places = 0;
          for (int &r : rows) places = std::exchange(r, places) + places;
          for (auto &g : groups) open[size_t(g.tb)] = rows[size_t(root(g.tb))];
          for (auto &g : groups) head[size_t(g.tb)] = open[size_t(g.tb)];
          open.assign(size_t(places), -1);
        }
        std::vector<double> cost;  // of a piece
        std::vector<int> of(n);    // a unit's piece
        const double total = std::accumulate(ucost.begin(), ucost.end(), 0.0);
        for (size_t i = 0; i < n; ++i) {
          int &q = open[size_t(head[size_t(units[i].tbeg)] + (best == kSkinny ? units[i].m0 / tbm : 0))];
          if (q < 0 || cost[size_t(q)] + ucost[i] > total / 24) {
            q = int(cost.size());
            cost.push_back(0.0);
          }
          cost[size_t(q)] += ucost[i];
          of[i] = q;
        }
        std::vector<int> order(cost.size()), xcd(cost.size()), turn(n);
        std::iota(order.begin(), order.end(), 0);
        std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return cost[size_t(a)] > cost[size_t(b)]; });
        std::array<double, kXcds> load{};
        for (int q : order) {
          const auto x = std::min_element(load.begin(), load.end());
          xcd[size_t(q)] = int(x - load.begin());
          *x += cost[size_t(q)];
        }
        std::iota(turn.begin(), turn.end(), 0);
        if (best == kSkinny) {  // a piece's units one after another
          std::vector<int> place(cost.size() + 1, 0);
          for (int q : of) ++place[size_t(q)];
          int sum = 0;
          for (int q : order) sum += std::exchange(place[size_t(q)], sum);
          for (size_t i = 0; i < n; ++i) turn[size_t(place[size_t(of[i])]++)] = int(i);
        }
        for (int i : turn) lists[size_t(xcd[size_t(of[size_t(i)])])].push_back(units[size_t(i)]);
        std::array<size_t, kXcds> at{};
        for (size_t i = 0; i < n; ++i) {
          size_t x = i % kXcds;
          for (size_t y = 0; at[x] == lists[x].size(); ++y) x = y;  // its list is used up: the next units of another
          su.push_back(lists[x][at[x]++]);
        }
      }
      units.swap(su);
    }
    auto *p = new itx_plan();
    p->prec = prec;
    p->tile = best;
    p->a_kcontig = akc;
    p->split_ok = first_kc;
    p->b_kcontig = bkc;
    p->ntasks = int(vt.size());
    p->nunits = int(units.size());
    p->flops = flops;
    const int occ = best == kSkinny && tinyq ? kSkinnyQOcc : tile_occupancy(best, prec, akc, bkc);
    p->grid = int(std::min<int64_t>(int64_t(units.size()), int64_t(cus) * occ));
    p->vec = (akc && bkc) ? vecbits : 0;
    const Skinny sk{maxN, tinyq, st.size() == groups.size() && maxK <= 4 * SK_KS ? (maxK + 3) / 4 : 0};
    // Small blocks of the reduced forms with short tasks: lanes along the rows
    // also where k is contiguous.  Along k most would idle (23 blocks of up to 60
    // x 15, K <= 8, BF16x3 6.2 and 9.3 us; block-sparse chain at chi = 110, K <=
    // 8, BF16x3 33.6 and 34.5).  Above 24 k it depends on the number of rows: the
    // chain at chi = 400 (K <= 28) 48.4 and 49.7 us, 52 blocks of up to 42 x 42 x
    // 42 13.8 and 12.5.
    const bool rows_only = best == kSmall && prec != ITX_PREC_F64 && maxK <= 24;
    p->fn = kernel_of(best, prec, akc && !rows_only, bkc && !rows_only, &p->block, p->vec, false, sk);
    p->fn_scalar = kernel_of(best, prec, akc && !rows_only, bkc && !rows_only, &p->block, 0, false, sk);
    p->nred = int(red.size());
    if (p->nred) {
      p->fn_red = best == kPipe64 ? reinterpret_cast<const void *>(&k_reduce_tiles<64, 64>)
                                  : reinterpret_cast<const void *>(&k_reduce_tiles<SM_M, SM_N>);
      p->grid_red = int(std::min<int64_t>(int64_t(red.size()) * (slot_elems / SM_T), int64_t(cus) * 8));
    }
    if (std::getenv("ITX_PLAN_LOG"))
      std::fprintf(stderr, "[itx plan] tasks=%d units=%d tile=%dx%d%s grid=%d akc=%d bkc=%d flops=%.3e split=%d\n",
                   p->ntasks, p->nunits, tbm, tbn, best == kSkinny ? "(skinny)" : best == kSmall ? "(small)" : "",
                   p->grid, int(akc), int(bkc), flops, p->nred);
    if (p->nunits > 0) {
      size_t bt_bytes = vt.size() * sizeof(GemmTask);
      size_t bu_bytes = units.size() * sizeof(WorkUnit);
      size_t br_bytes = red.size() * sizeof(WorkUnit);
      size_t o_units = (bt_bytes + 255) & ~size_t(255);
      size_t o_red = (o_units + bu_bytes + 255) & ~size_t(255);
      size_t o_tab = (o_red + br_bytes + 255) & ~size_t(255);
      size_t o_ws = (o_tab + tab.size() * sizeof(int64_t) + 255) & ~size_t(255);
      size_t total = o_ws + sizeof(double) * size_t(nslots) * slot_elems;
      // the device image: tasks | units | reduction units | tables, each
      // 256-byte aligned, assembled in the staging arena
      const UploadPart parts[4] = {{vt.data(), 0, bt_bytes},
                                   {units.data(), o_units, bu_bytes},
                                   {red.data(), o_red, br_bytes},
                                   {tab.data(), o_tab, tab.size() * sizeof(int64_t)}};
      int rc3 = ITX_OK;
      if (into) {
        if (total > into_cap) {
          delete p;
          return set_err(ctx, ITX_ERR_UNSUPPORTED,
                         "contraction: the plan needs " + std::to_string(total) + " bytes of device memory, more than the " +
                             std::to_string(into_cap) + "-byte scratch of the allocation-free entry point");
        }
        p->dev = into;
        p->own_dev = false;
      } else {
        rc3 = pool_alloc(ctx, total, &p->dev);
        if (rc3) {
          delete p;
          return rc3;
        }
      }
      p->ctx = ctx;
      rc3 = stage_upload_parts(ctx, p->dev, parts, 4, o_ws);
      if (rc3) {
        if (p->own_dev) pool_free(ctx, p->dev);
        delete p;
        return rc3;
      }
      p->dev_bytes = total;
      p->d_tasks = reinterpret_cast<const GemmTask *>(p->dev);
      p->d_units = reinterpret_cast<const WorkUnit *>(static_cast<char *>(p->dev) + o_units);
      p->d_tab = reinterpret_cast<const int64_t *>(static_cast<char *>(p->dev) + o_tab);
      if (p->nred) {
        p->d_red = reinterpret_cast<const WorkUnit *>(static_cast<char *>(p->dev) + o_red);
        p->ws = reinterpret_cast<double *>(static_cast<char *>(p->dev) + o_ws);
      }
    }
    ctx->plans.insert(p);
    *pout = p;
    return ITX_OK;
  };

  // ---- tile selection ------------------------------------------------
  // Narrow tasks (all N <= 32, K <= 64) over large C blocks take the skinny
  // kernels, C blocks of at most 8192 elements (small QN blocks) the
  // small-block kernels.  Otherwise, in order: ITX_FORCE_TILE, the tuning
  // table entry of this size class, a measurement of every MFMA tile when
  // autotuning is on (result stored in the table), else a cost model.
  int best = 0;
  const std::string key = tune_key(prec, akc, bkc, maxM, maxN, maxKsum, int(groups.size()));
  const char *force = std::getenv("ITX_FORCE_TILE");
  double rows = 0;
  for (auto &g : groups) rows += g.M;
  const double avg_rows = groups.empty() ? 0.0 : rows / double(groups.size());
  const bool narrow = maxN <= SK_N && maxK <= SK_K;
  // FP64: the eight waves of a small-block unit share its k, and wait for
  // each other, so they want more than four chunks of 16 k, and no more units
  // than CUs (block-sparse chain, 32 x 32 tiles against small blocks: chi =
  // 250 first stage, 1.5 chunks, 4.7 and 7.1 us; chi = 500 last stage, 14
  // chunks of 156 tiles, 13.0 and 11.0; chi = 750, 19 of 326, 18.4 and 19.8)
  double n32 = 0, chunks = 0;
  for (auto &g : groups) {
    const double n = double((g.M + 31) / 32) * double((g.N + 31) / 32);
    n32 += n;
    for (int t = g.tb; t < g.te; ++t) chunks += n * double((st[t].K + 15) / 16);
  }
  const bool long_k = prec != ITX_PREC_F64 || (chunks > 4 * n32 && n32 <= cus);
  // what a forced tile or a table entry must meet; an entry is shared by all
  // sizes of its class, aligned and not
  auto usable = [&](int t) { return t >= 0 && t < kNumTiles && (t != kSkinny || narrow) && tile_ok(t); };
  const auto tuned = ctx->tune.find(key);
  if (!st.empty() && !force && narrow && avg_rows >= 256) {
    best = kSkinny;
  } else if (!st.empty() && !force && double(maxM) * double(maxN) <= 8192.0) {
    best = long_k ? kSmall : 4;
  } else if (force) {
    best = std::atoi(force);
    if (!usable(best)) best = 0;
  } else if (tuned != ctx->tune.end() && usable(tuned->second)) {
    best = tuned->second;
  } else if (ctx->autotune && !into && !st.empty()) {
    void *bufA = nullptr, *bufB = nullptr, *bufC = nullptr;
    int rc2 = pool_alloc(ctx, sizeof(double) * size_t(extA), &bufA);
    if (!rc2) rc2 = pool_alloc(ctx, sizeof(double) * size_t(extB), &bufB);
    if (!rc2) rc2 = pool_alloc(ctx, sizeof(double) * size_t(extC), &bufC);
    if (rc2) return rc2;
    itx_fill(ctx, static_cast<double *>(bufA), size_t(extA), 0.0);
    itx_fill(ctx, static_cast<double *>(bufB), size_t(extB), 0.0);
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    float best_ms = 1e30f;
    for (int ti = 0; ti < kNumTiles; ++ti) {
      if (ti == kSkinny || ti == kSmall) continue;
      // in FP64 the kernel of kPipe128, which takes any alignment
      if (prec == ITX_PREC_F64 && (ti == kDgemm || ti == kDgemm2)) continue;
      itx_plan *pc = nullptr;
      if (finalize(ti, &pc)) continue;
      const double *A = static_cast<const double *>(bufA), *B = static_cast<const double *>(bufB);
      double *Cp = static_cast<double *>(bufC);
      launch_plan(ctx, pc, A, B, Cp, 1.0, 0.0);
      (void)hipEventRecord(e0, ctx->stream);
      for (int r = 0; r < 3; ++r) launch_plan(ctx, pc, A, B, Cp, 1.0, 0.0);
      (void)hipEventRecord(e1, ctx->stream);
      (void)hipEventSynchronize(e1);
      float ms = 0;
      (void)hipEventElapsedTime(&ms, e0, e1);
      if (ms < best_ms) {
        best_ms = ms;
        best = ti;
      }
      itx_plan_destroy(ctx, pc);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    pool_free(ctx, bufA);
    pool_free(ctx, bufB);
    pool_free(ctx, bufC);
    ctx->tune[key] = best;
  } else {
    if (prec == ITX_PREC_F32 && dg_ok) {
      // Tile 14 where this model of the unpipelined tiles prefers it: it sums
      // in another order than the rest.
      double best_t = 1e300;
      for (int ti : {0, 1, 2, 3, 4, 6, 7, 8, 9, kDgemm}) {
        const TileCfg ts = kTiles[ti];
        std::vector<double> costs;
        int64_t n = 0;
        double one = 0;
        for (auto &g : groups) {
          const int64_t tiles = int64_t((g.M + ts.bm - 1) / ts.bm) * ((g.N + ts.bn - 1) / ts.bn);
          one = double(ts.bm) * ts.bn * (g.ksum + BK * (g.te - g.tb) + 8);
          n += tiles;
          if (groups.size() > 1) costs.insert(costs.end(), size_t(tiles), one);
        }
        if (!n) continue;
        // workgroups resident per CU: the tile's occupancy, or fewer when the
        // units do not fill that many slots (a CU running one workgroup does not
        // run it `occupancy` times slower; without this the FP32 form picked a
        // 64 x 256 tile for 150 units of the chi = 1024 QN chain, 86 us against
        // 40 us)
        const int occ = int(std::max<int64_t>(
            1, std::min<int64_t>(tile_occupancy(ti, prec, akc, bkc), (n + cus - 1) / cus)));
        const int64_t slots = int64_t(cus) * occ;
        const double tt = (costs.empty() ? lpt_makespan(n, one, slots) : lpt_makespan(costs, slots)) * occ / ts.eff32;
        if (tt < best_t * 0.97) {
          best_t = tt;
          best = ti;
        }
      }
    }
    // The pipelined tiles (k_pipe) and the 32 x 32 tile.  A unit costs its k
    // stages of 16 and a few more for every task and for itself; `alone` is
    // the time of a stage (us) of a workgroup that has its CU to itself,
    // `shared` the CU's time per stage when it has several, by layout: both
    // operands contiguous along k; each along k or in runs of 16 rows; others.
    // Fitted to the stages of the dense chain at chi = 48 to 1024 and to products
    // of 600 to 4000 rows and columns with K = 8 to 1151; the last layout to its
    // MPO stage at d = 4, k = 18, where the operator is read in single strided
    // elements.  One class for the last two took 128 x 128 where 64 x 64 is
    // better: 3362 x 1159 x 32 along rows 21.5 and 12.7 us in FP32, 20 and 13 in
    // BF16x3, 1500 x 1500 x 200 37 and 29 in FP64.
    // FP64, us as 32 x 32, 64 x 64, 128 x 128: last stage, chi = 255 43, 28
    // (split eight ways), 168; chi = 512 152, 96, 293; chi = 1024 1040, 660,
    // 593; MPO stage, chi = 32 21.6, 18.4, 50.6; chi = 330 1274, 676, 574.
    // FP32, and 32 x 64 (before: 64 x 64 of k_gemm): last stage, chi = 256 37,
    // 35.4, 91.5, 28.4 (69); chi = 512 139, 77, 177, 77 (134); chi = 1024 876,
    // 440, 358, 516 (579).  BF16x3 (before: 64 x 64 of k_gemm3): chi = 256 23,
    // 26, 53 (43); chi = 512 87, 53, 107 (85); chi = 1024 600, 315, 210 (343).
    struct Model {
      int tile, bm, bn;
      double per_task, per_unit;
      double alone[3], shared[3];  // by layout: along k, along k or rows, other
    };
    const bool vector = prec == ITX_PREC_BF16X3 ? vecbits & 2 : vecbits & 1;
    const double v1 = vector ? 1.0 : prec == ITX_PREC_F64 ? 1.1 : prec == ITX_PREC_F32 ? 1.2 : 1.6;  // single loads
    const double w1 = vector ? 1.0 : prec == ITX_PREC_F64 ? 1.2 : prec == ITX_PREC_F32 ? 1.25 : 1.4;  // of 32 x 32
    const double s4 = maxK > 2048 ? 0.28 : 0.22;  // with long k its operands leave the L2
    const int lay = akc && bkc ? 0 : run_work > 0 ? 1 : 2;
    const bool dear = lay < 2;  // a unit's own time: behind the slow stages of the last layout it is short
    const Model f64[] = {{4, 32, 32, 1, 1, {0.45 * w1, 0.50, 0.50}, {s4 * w1, 0.27, 0.50}},
                         {kPipe64, 64, 64, 3, dear ? 1.0 : 2.0, {0.56, 0.64, 0.70}, {0.50 * v1, 0.54, 0.88}},
                         {kPipe128, 128, 128, 2, dear ? 1.5 : 1.0, {1.87 * v1, 2.00, 2.65}, {1.87 * v1, 2.05, 2.65}}};
    const Model f32[] = {{4, 32, 32, 1, 1, {0.42 * w1, 0.45, 0.50}, {0.18 * w1, 0.24, 0.50}},
                         {kPipe32, 32, 64, 2, dear ? 3.0 : 1.0, {0.28 * v1, 0.40, 0.75}, {0.21 * v1, 0.27, 0.85}},
                         {kPipe64, 64, 64, 3, 2, {0.43 * v1, 0.45, 0.62}, {0.33 * v1, 0.37, 0.83}},
                         {kPipe128, 128, 128, 2, dear ? 3.0 : 1.0, {1.13 * v1, 1.31, 1.80}, {1.13 * v1, 1.40, 2.05}}};
    const Model bf[] = {{4, 32, 32, 1, dear ? 3.0 : 1.0, {0.28 * w1, 0.42, 0.45}, {0.14 * w1, 0.23, 0.37}},
                        {kPipe64, 64, 64, 3, dear ? 3.0 : 2.0, {0.31 * v1, 0.49, 0.70}, {0.235 * v1, 0.30, 0.73}},
                        {kPipe128, 128, 128, 2, dear ? 4.0 : 1.0, {0.65 * v1, 0.95, 1.65}, {0.74 * v1, 1.00, 1.90}}};
    const Model *models = prec == ITX_PREC_F64 ? f64 : prec == ITX_PREC_F32 ? f32 : bf;
    const size_t nm = best == kDgemm ? 0 : prec == ITX_PREC_F32 ? std::size(f32) : std::size(f64);
    if (nm) best = 4;
    double best_t = 1e300;
    for (const Model *md = models; md < models + nm; ++md) {
      std::vector<double> costs;
      int64_t n = 0;
      double most = 0;
      const int ns = md->tile == kPipe64 ? pipe_split() : 1;
      for (auto &g : groups) {
        double c = md->per_unit;
        for (int t = g.tb; t < g.te; ++t) c += double((st[t].K + DG_BK - 1) / DG_BK) / ns + md->per_task;
        const int64_t tiles = int64_t((g.M + md->bm - 1) / md->bm) * ((g.N + md->bn - 1) / md->bn) * ns;
        most = std::max(most, c);
        n += tiles;
        if (groups.size() > 1) costs.insert(costs.end(), size_t(tiles), c);
      }
      double tt = most * md->alone[lay];
      if (n > cus)
        tt = std::max(tt, (costs.empty() ? lpt_makespan(n, most, cus) : lpt_makespan(costs, cus)) * md->shared[lay]);
      if (ns > 1)  // the partial tiles and the second launch
        tt += 5.0 + double(ns) * groups[0].M * groups[0].N * 16.0 / 4e6;
      if (tt < best_t) {
        best_t = tt;
        best = md->tile;
      }
    }
    if (prec == ITX_PREC_F64 && st.size() == 1 && st[0].K <= 640) {  // above, its partial tiles cost more
      const bool fine = n32 < cus / 2;  // as finalize sizes the units
      const double n16 = double((st[0].M + 15) / 16) * double((st[0].N + 15) / 16);
      if ((fine ? n16 : n32) <= cus && 2.0 + (fine ? 1.35 : 2.2) * ((st[0].K + 127) / 128) < best_t) best = kSmall;
    }
  }
  rc = finalize(best, out);
  // The plan of the ordinary call, and so its sums, wherever the caller's
  // scratch holds it; else without partial tiles, then in larger units.
  if (rc == ITX_ERR_UNSUPPORTED && into) {
    lean = true;
    rc = finalize(best, out);
    const bool small = double(maxM) * double(maxN) <= 8192.0;
    if (rc == ITX_ERR_UNSUPPORTED && !force && best != kSkinny && !(small && best == kSmall))
      rc = finalize(small ? kSmall : kPipe128, out);
  }
  return rc;
}

const void *plan_fn(const itx_plan *p, const double *A, const double *B) {
  // the vector-load kernel reads 16-byte pairs (or quads of split words):
  // its operands must be 16-byte aligned (caching-pool blocks are 256-byte
  // aligned)
  const bool aligned = ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15) == 0;
  return (p->vec && aligned) ? p->fn : p->fn_scalar;
}

KernelArgs plan_args(const itx_plan *p, int which, const double *A, const double *B, double *C, double alpha,
                     double beta) {
  if (which == 0)  // the contraction (into the workspace when split)
    return KernelArgs{A, B, p->nred ? p->ws : C, p->d_tasks, p->d_units, p->nunits, p->d_tab, alpha, beta};
  return KernelArgs{p->ws, nullptr, C, p->d_tasks, p->d_red, p->nred, p->d_tab, alpha, beta};
}

int launch_plan(itx_ctx *ctx, const itx_plan *p, const double *A, const double *B, double *C, double alpha,
                double beta) {
  if (!p) return set_err(ctx, ITX_ERR_ARG, "null plan");
  if (p->nunits == 0) return ITX_OK;
  void *args[KernelArgs::kCount];
  KernelArgs ka = plan_args(p, 0, A, B, C, alpha, beta);
  ka.pointers(args);
  ITX_CHECK_HIP(ctx, hipLaunchKernel(plan_fn(p, A, B), dim3(p->grid), dim3(p->block), args, 0, ctx->stream));
  if (p->nred) {
    KernelArgs kr = plan_args(p, 1, A, B, C, alpha, beta);
    kr.pointers(args);
    ITX_CHECK_HIP(ctx, hipLaunchKernel(p->fn_red, dim3(p->grid_red), dim3(SM_T_RED), args, 0, ctx->stream));
  }
  return ITX_OK;
}

namespace {

std::string plan_key(const char *kind, int rA, const int32_t *labA, int rB, const int32_t *labB, int rC,
                     const int32_t *labC, int ntasks, const int64_t *offs, const int64_t *blkA,
                     const int64_t *blkB, int prec) {
  std::string k;
  k.reserve(64 + 8 * (rA + rB + rC) + size_t(ntasks) * 8 * (3 + rA + rB));
  auto put = [&](const void *d, size_t n) { k.append(static_cast<const char *>(d), n); };
  put(kind, std::strlen(kind));
  put(&rA, sizeof rA);
  put(&rB, sizeof rB);
  put(&rC, sizeof rC);
  put(&prec, sizeof prec);
  put(&ntasks, sizeof ntasks);
  put(labA, sizeof(int32_t) * rA);
  put(labB, sizeof(int32_t) * rB);
  put(labC, sizeof(int32_t) * rC);
  put(offs, sizeof(int64_t) * 3 * size_t(ntasks));
  put(blkA, sizeof(int64_t) * rA * size_t(ntasks));
  put(blkB, sizeof(int64_t) * rB * size_t(ntasks));
  return k;
}

constexpr size_t kPlanCacheMax = 96;

int cached_plan(itx_ctx *ctx, const std::string &key, itx_plan **out,
                const std::function<int(itx_plan **)> &make) {
  auto it = ctx->plan_cache.find(key);
  if (it != ctx->plan_cache.end()) {
    *out = it->second;
    return ITX_OK;
  }
  itx_plan *p = nullptr;
  int rc = make(&p);
  if (rc) return rc;
  if (ctx->plan_cache.size() >= kPlanCacheMax) {
    // evict the oldest entry (FIFO); its device block returns to the
    // stream-ordered pool, so kernels already enqueued still read it intact
    const std::string old = ctx->plan_lru.front();
    ctx->plan_lru.erase(ctx->plan_lru.begin());
    auto jt = ctx->plan_cache.find(old);
    if (jt != ctx->plan_cache.end()) {
      itx_plan_destroy(ctx, jt->second);
      ctx->plan_cache.erase(jt);
    }
  }
  ctx->plan_cache[key] = p;
  ctx->plan_lru.push_back(key);
  *out = p;
  return ITX_OK;
}

}  // namespace
}  // namespace itx

extern "C" {

int itx_plan_dense(itx_ctx *ctx, int rA, const int64_t *dimsA, const int32_t *labA, int rB,
                   const int64_t *dimsB, const int32_t *labB, int rC, const int64_t *dimsC,
                   const int32_t *labC, int prec, itx_plan **out) {
  if (!ctx || !out) return ITX_ERR_ARG;
  const int64_t offs[3] = {0, 0, 0};
  return itx::build_plan(ctx, rA, labA, rB, labB, rC, labC, 1, offs, dimsA, dimsB, dimsC, prec, out);
}

int itx_plan_qn(itx_ctx *ctx, int rA, const int32_t *labA, int rB, const int32_t *labB, int rC,
                const int32_t *labC, int ntasks, const int64_t *offs, const int64_t *blkdimsA,
                const int64_t *blkdimsB, int prec, itx_plan **out) {
  if (!ctx || !out) return ITX_ERR_ARG;
  return itx::build_plan(ctx, rA, labA, rB, labB, rC, labC, ntasks, offs, blkdimsA, blkdimsB, nullptr, prec,
                         out);
}

int itx_plan_execute(itx_ctx *ctx, const itx_plan *plan, const double *A, const double *B, double *C,
                     double alpha, double beta) {
  if (!ctx) return ITX_ERR_ARG;
  return itx::launch_plan(ctx, plan, A, B, C, alpha, beta);
}

double itx_plan_flops(const itx_plan *plan) { return plan ? plan->flops : 0.0; }

int itx_split_bf16(itx_ctx *ctx, const double *x, uint32_t *y, size_t n) {
  if (!ctx || (n && (!x || !y))) return ITX_ERR_ARG;
  if (n == 0) return ITX_OK;
  const unsigned grid = unsigned(std::min<size_t>((n + 255) / 256, size_t(ctx->num_cus) * 16));
  hipLaunchKernelGGL(itx::k_split_bf16, dim3(grid), dim3(256), 0, ctx->stream, x, y, n);
  ITX_CHECK_HIP(ctx, hipGetLastError());
  return ITX_OK;
}

int itx_plan_set_split(itx_ctx *ctx, itx_plan *plan, int on) {
  if (!ctx || !plan) return ITX_ERR_ARG;
  const bool want = on != 0;
  if (want == bool(plan->split)) return ITX_OK;
  if (want && (plan->prec != ITX_PREC_BF16X3 || plan->tile == itx::kSkinnyTile || plan->tile == 10 ||
               !plan->split_ok || plan->nred))
    return itx::set_err(ctx, ITX_ERR_UNSUPPORTED,
                        "itx_plan_set_split: pre-split operands need a BF16x3 MFMA plan with both operands "
                        "contiguous along the contracted index");
  plan->split = want ? 1 : 0;
  if (plan->nunits > 0) {
    const bool akc = plan->a_kcontig, bkc = plan->b_kcontig;
    if (want) {
      plan->fn = itx::kernel_of(plan->tile, plan->prec, akc, bkc, &plan->block, plan->vec & 4 ? 4 : 0, true);
      plan->fn_scalar = itx::kernel_of(plan->tile, plan->prec, akc, bkc, &plan->block, 0, true);
    } else {
      plan->fn = itx::kernel_of(plan->tile, plan->prec, akc, bkc, &plan->block, plan->vec);
      plan->fn_scalar = itx::kernel_of(plan->tile, plan->prec, akc, bkc, &plan->block, 0);
    }
  }
  return ITX_OK;
}

int itx_plan_info(const itx_plan *plan, int *tile, int *form, int *ntasks, int *nunits) {
  if (!plan) return ITX_ERR_ARG;
  // the skinny path is HBM-bound and computes in FP64 in every form
  const int f = plan->tile == itx::kSkinnyTile ? ITX_PREC_F64 : plan->prec;
  if (tile) *tile = plan->tile;
  if (form) *form = f;
  if (ntasks) *ntasks = plan->ntasks;
  if (nunits) *nunits = plan->nunits;
  return ITX_OK;
}

int itx_plan_destroy(itx_ctx *ctx, itx_plan *plan) {
  if (!plan) return ITX_OK;
  // the device block goes back to the context's stream-ordered pool (no
  // wait); without a context it stays with the pool until itx_destroy
  if (ctx) {
    if (plan->dev && plan->own_dev) itx::pool_free(ctx, plan->dev);
    ctx->plans.erase(plan);
  }
  delete plan;
  return ITX_OK;
}

int itx_chain_create(itx_ctx *ctx, int nstages, itx_plan *const *plans, itx_chain **out) {
  if (!ctx || !out || nstages <= 0 || !plans) return ITX_ERR_ARG;
  *out = nullptr;
  for (int i = 0; i < nstages; ++i)
    if (!plans[i]) return itx::set_err(ctx, ITX_ERR_ARG, "itx_chain_create: null plan");
  auto *ch = new itx_chain();
  ch->plans.assign(plans, plans + nstages);
  ch->args.resize(2 * size_t(nstages));
  ch->nodes.assign(2 * size_t(nstages), nullptr);
  ch->funcs.assign(2 * size_t(nstages), nullptr);
  ctx->chains.insert(ch);
  *out = ch;
  return ITX_OK;
}

int itx_chain_launch(itx_ctx *ctx, itx_chain *ch, const double *const *A, const double *const *B,
                     double *const *C, const double *alpha, const double *beta) {
  if (!ctx || !ch || !A || !B || !C) return ITX_ERR_ARG;
  const int n = int(ch->plans.size());
  // node 2i: the contraction of stage i; node 2i+1: its reduction pass
  auto args_of = [&](int x) {
    const int i = x / 2;
    return itx::plan_args(ch->plans[size_t(i)], x % 2, A[i], B[i], C[i], alpha ? alpha[i] : 1.0,
                          beta ? beta[i] : 0.0);
  };
  auto active = [&](int x) {
    const itx_plan *p = ch->plans[size_t(x / 2)];
    return p->nunits > 0 && (x % 2 == 0 || p->nred > 0);
  };
  auto fn_of = [&](int x) {
    const itx_plan *p = ch->plans[size_t(x / 2)];
    return x % 2 ? p->fn_red : itx::plan_fn(p, A[x / 2], B[x / 2]);
  };
  if (ch->exec) {
    // a changed operand alignment changes a stage's kernel: rebuild
    bool same = true;
    for (int x = 0; x < 2 * n && same; ++x)
      if (ch->nodes[size_t(x)] && fn_of(x) != ch->funcs[size_t(x)]) same = false;
    if (!same) {
      hipGraphExecDestroy(ch->exec);
      hipGraphDestroy(ch->graph);
      ch->exec = nullptr;
      ch->graph = nullptr;
      ch->nodes.assign(ch->nodes.size(), nullptr);
    }
  }
  auto params_of = [&](int x, void **argv) {
    hipKernelNodeParams kp{};
    const itx_plan *p = ch->plans[size_t(x / 2)];
    ch->funcs[size_t(x)] = fn_of(x);
    kp.func = const_cast<void *>(ch->funcs[size_t(x)]);
    kp.gridDim = dim3(unsigned(x % 2 ? p->grid_red : p->grid));
    kp.blockDim = dim3(unsigned(x % 2 ? itx::SM_T_RED : p->block));
    kp.sharedMemBytes = 0;
    ch->args[size_t(x)].pointers(argv);
    kp.kernelParams = argv;
    kp.extra = nullptr;
    return kp;
  };
  if (!ch->exec) {
    // first launch: one kernel node per launch, each after the previous
    // one (the stream order of the eager path)
    ITX_CHECK_HIP(ctx, hipGraphCreate(&ch->graph, 0));
    hipGraphNode_t prev = nullptr;
    for (int x = 0; x < 2 * n; ++x) {
      ch->args[size_t(x)] = args_of(x);
      if (!active(x)) continue;
      void *argv[itx::KernelArgs::kCount];
      hipKernelNodeParams kp = params_of(x, argv);
      ITX_CHECK_HIP(ctx, hipGraphAddKernelNode(&ch->nodes[size_t(x)], ch->graph, prev ? &prev : nullptr,
                                               prev ? 1 : 0, &kp));
      prev = ch->nodes[size_t(x)];
    }
    ITX_CHECK_HIP(ctx, hipGraphInstantiate(&ch->exec, ch->graph, nullptr, nullptr, 0));
  } else {
    // replay: patch the nodes whose operands or scalars changed
    for (int x = 0; x < 2 * n; ++x) {
      if (!ch->nodes[size_t(x)]) continue;
      const itx::KernelArgs a = args_of(x);
      itx::KernelArgs &c = ch->args[size_t(x)];
      if (a.A == c.A && a.B == c.B && a.C == c.C && a.alpha == c.alpha && a.beta == c.beta) continue;
      c = a;
      void *argv[itx::KernelArgs::kCount];
      hipKernelNodeParams kp = params_of(x, argv);
      ITX_CHECK_HIP(ctx, hipGraphExecKernelNodeSetParams(ch->exec, ch->nodes[size_t(x)], &kp));
    }
  }
  ITX_CHECK_HIP(ctx, hipGraphLaunch(ch->exec, ctx->stream));
  return ITX_OK;
}

int itx_chain_destroy(itx_ctx *ctx, itx_chain *ch) {
  if (!ch) return ITX_OK;
  if (ctx) {
    hipStreamSynchronize(ctx->stream);
    ctx->chains.erase(ch);
  }
  if (ch->exec) hipGraphExecDestroy(ch->exec);
  if (ch->graph) hipGraphDestroy(ch->graph);
  delete ch;
  return ITX_OK;
}

int itx_contract_dense(itx_ctx *ctx, const double *A, int rA, const int64_t *dimsA, const int32_t *labA,
                       const double *B, int rB, const int64_t *dimsB, const int32_t *labB, double *C, int rC,
                       const int64_t *dimsC, const int32_t *labC, double alpha, double beta, int prec) {
  if (!ctx) return ITX_ERR_ARG;
  const int64_t offs[3] = {0, 0, 0};
  std::string key = itx::plan_key("D", rA, labA, rB, labB, rC, labC, 1, offs, dimsA, dimsB, prec);
  key.append(reinterpret_cast<const char *>(dimsC), sizeof(int64_t) * rC);
  itx_plan *p = nullptr;
  int rc = itx::cached_plan(ctx, key, &p, [&](itx_plan **o) {
    return itx::build_plan(ctx, rA, labA, rB, labB, rC, labC, 1, offs, dimsA, dimsB, dimsC, prec, o);
  });
  if (rc) return rc;
  return itx::launch_plan(ctx, p, A, B, C, alpha, beta);
}

int itx_contract_qn(itx_ctx *ctx, const double *A, int rA, const int32_t *labA, const double *B, int rB,
                    const int32_t *labB, double *C, int rC, const int32_t *labC, int ntasks,
                    const int64_t *offs, const int64_t *blkdimsA, const int64_t *blkdimsB, double alpha,
                    int prec) {
  if (!ctx) return ITX_ERR_ARG;
  std::string key = itx::plan_key("Q", rA, labA, rB, labB, rC, labC, ntasks, offs, blkdimsA, blkdimsB, prec);
  itx_plan *p = nullptr;
  int rc = itx::cached_plan(ctx, key, &p, [&](itx_plan **o) {
    return itx::build_plan(ctx, rA, labA, rB, labB, rC, labC, ntasks, offs, blkdimsA, blkdimsB, nullptr, prec,
                           o);
  });
  if (rc) return rc;
  return itx::launch_plan(ctx, p, A, B, C, alpha, 0.0);
}

int itx_contract_qn_noalloc(itx_ctx *ctx, const double *A, int rA, const int32_t *labA, const double *B, int rB,
                            const int32_t *labB, double *C, int rC, const int32_t *labC, int ntasks,
                            const int64_t *offs, const int64_t *blkdimsA, const int64_t *blkdimsB, double alpha,
                            int prec) {
  if (!ctx) return ITX_ERR_ARG;
  if (!ctx->scratch) return itx::set_err(ctx, ITX_ERR_UNSUPPORTED, "itx_contract_qn_noalloc: no scratch address");
  // the plan lives in host memory for this call only; its device block is
  // the scratch array, which the stream reuses in order for the next call
  itx_plan *p = nullptr;
  int rc = itx::build_plan(ctx, rA, labA, rB, labB, rC, labC, ntasks, offs, blkdimsA, blkdimsB, nullptr, prec, &p,
                           ctx->scratch, ctx->scratch_bytes);
  if (rc) return rc;
  rc = itx::launch_plan(ctx, p, A, B, C, alpha, 0.0);
  itx_plan_destroy(ctx, p);
  return rc;
}

}  // extern "C"

extern "C" {

int itx_set_autotune(itx_ctx *ctx, int on) {
  if (!ctx) return ITX_ERR_ARG;
  ctx->autotune = on ? 1 : 0;
  return ITX_OK;
}

int itx_tune_save(itx_ctx *ctx, const char *path) {
  if (!ctx || !path) return ITX_ERR_ARG;
  std::ofstream f(path);
  if (!f) return itx::set_err(ctx, ITX_ERR_ARG, std::string("itx_tune_save: cannot write ") + path);
  for (auto &kv : ctx->tune) f << kv.first << '|' << kv.second << '\n';
  return ITX_OK;
}

int itx_tune_load(itx_ctx *ctx, const char *path) {
  if (!ctx || !path) return ITX_ERR_ARG;
  std::ifstream f(path);
  if (!f) return itx::set_err(ctx, ITX_ERR_ARG, std::string("itx_tune_load: cannot read ") + path);
  std::string line;
  while (std::getline(f, line)) {
    auto bar = line.find('|');
    if (bar == std::string::npos) continue;
    ctx->tune[line.substr(0, bar)] = std::atoi(line.c_str() + bar + 1);
  }
  return ITX_OK;
}

int itx_tune_size(itx_ctx *ctx) { return ctx ? int(ctx->tune.size()) : 0; }

}  // extern "C"
