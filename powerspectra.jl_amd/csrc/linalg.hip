// FP64 LU decoupling: `lu` and `A \ B` (reference
// src/blockspectralmatrix.jl:89-129) and decouple_covmat
// (src/covariance.jl:8-14).  Julia's `lu` is LAPACK getrf with partial
// pivoting and throws SingularException on an exact zero pivot.  The
// factorisation is this file's blocked getrf (HIP leaf kernels + rocBLAS
// updates) in LAPACK layout; right-hand sides at hand move their rows with its
// panels, decouple_covmat's second ones by a gather (rocSOLVER's laswp above
// kPermMax rows), and this file's forward and back substitution follow (rocBLAS
// updates between diagonal blocks).
#include "psx_internal.h"

#include <utility>

#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

namespace psx {

static rocblas_handle blas(Ctx* c) {
  if (!c->blas) {
    rocblas_handle h;
    PSX_REQUIRE(rocblas_create_handle(&h) == rocblas_status_success, PSX_ERR_DEVICE,
                "rocblas_create_handle failed");
    rocblas_set_stream(h, c->stream);
    c->blas = h;
  }
  return static_cast<rocblas_handle>(c->blas);
}

void release_lanes(Ctx* c);

void release_blas(Ctx* c) {
  release_lanes(c);
  if (c->blas) {
    rocblas_destroy_handle(static_cast<rocblas_handle>(c->blas));
    c->blas = nullptr;
  }
}

#define PSX_ROC(call)                                                         \
  do {                                                                        \
    rocblas_status s_ = (call);                                               \
    PSX_REQUIRE(s_ == rocblas_status_success, PSX_ERR_DEVICE,                 \
                std::string(#call) + " failed: " + rocblas_status_to_string(s_)); \
  } while (0)

void dgemm_dev(Ctx* c, int m, int n, int k, const double* dA, int64_t lda, const double* dB,
               int64_t ldb, double* dC, int64_t ldc) {
  const double one = 1.0, zero = 0.0;
  PSX_ROC(rocblas_dgemm(blas(c), rocblas_operation_none, rocblas_operation_none, m, n, k, &one,
                        dA, (rocblas_int)lda, dB, (rocblas_int)ldb, &zero, dC,
                        (rocblas_int)ldc));
}

// ---- LU with partial pivoting ---------------------------------------------
// Right-looking blocked getrf.  Panels of kLuPanel columns end with their U rows
// (panel_trsm) and a trailing rocBLAS dgemm of depth kLuPanel.  Inside a panel, leaves
// of 8 to 32 columns are factored by one workgroup holding the leaf's rows in
// registers (lu_leaf_wg), or, above kLuWgRowsMax rows, one column per launch
// (lu_leaf_col).  Ties in |pivot| go to the smallest row index, NaN ranks
// first, and a zero pivot column is skipped and reported (first one, 1-based),
// as getrf does.  Within a leaf rows are not moved; after it the pivots become
// LAPACK's row interchanges (ipiv, 1-based) and the leaf's net row movement,
// applied to the panel's columns at once and to all others once per panel, as
// the panel's net movement: the matrix ends exactly as getrf's physical swaps
// leave it.  (A single cooperative launch per leaf with a grid barrier per
// column measured slower: the cross-XCD barrier costs more than a launch.)
constexpr int kLuLeaf = 32;
constexpr int kLuPanel = 256;
constexpr int kLuRows = 128;     // rows per workgroup of the multi-workgroup leaf kernels

struct LuWork {
  // per-workgroup pivot candidates, two buffers of cstride entries: the
  // launch for column j reads buffer j & 1 and writes the other, since the
  // workgroups of one launch read every candidate while others write theirs.
  // Each candidate is |value|, its row, and that row's entries from the
  // candidate's column to the leaf's end (kLuLeaf slots).
  double* candv;
  int* candi;
  double* candrow;
  int cstride;
  unsigned char* done;// rows already chosen as pivots in the current leaf
  int* piv;           // the leaf's pivot rows (original positions)
  int* ipiv;          // LAPACK interchanges, 1-based, n entries
  int* info;          // first zero pivot column (1-based) or 0
  // net row movements of the panel's leaves: position mkey[k] receives the row
  // at position mval[k]; the leaf at panel column d with nc columns has the
  // entries [2 d, 2 d + 2 nc), unused ones with key -1
  int* mkey;
  int* mval;
  // the panel's net movement as lu_panel_perm leaves it: entries [0, panel
  // width) are the panel's own rows, in order, the others rows below it
  int* pkey;
  int* pval;
  int* pcount;
};

// |x| for the pivot search; NaN ranks above everything, so a NaN column
// still yields a row (and propagates) and the search never comes back empty.
__device__ inline double lu_mag(double x) { return x != x ? INFINITY : fabs(x); }

__device__ inline void lu_better(double& v, int& r, double ov, int orr) {
  if (ov > v || (ov == v && orr < r)) {
    v = ov;
    r = orr;
  }
}

// (value, row) maximum with ties to the smaller row over the workgroup; every
// thread returns with the result.
__device__ inline void lu_argmax_block(double& v, int& r) {
  __shared__ double sv[kLuRows / 64];
  __shared__ int sr[kLuRows / 64];
  for (int o = 32; o >= 1; o >>= 1) lu_better(v, r, __shfl_xor(v, o), __shfl_xor(r, o));
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sv[w] = v;
    sr[w] = r;
  }
  __syncthreads();
  v = sv[0];
  r = sr[0];
  for (int k = 1; k < kLuRows / 64; ++k) lu_better(v, r, sv[k], sr[k]);
}

// Publish the workgroup's candidate into buffer `buf`: the winning thread
// copies its row entries vals[first .. first+count).
__device__ inline void lu_publish(const LuWork& w, int buf, double v, int r, int i,
                                  const double* vals, int first, int count) {
  const int slot = buf * w.cstride + (int)blockIdx.x;
  if (threadIdx.x == 0) {
    w.candv[slot] = v;
    w.candi[slot] = r;
  }
  if (i == r) {
    double* dst = w.candrow + (int64_t)slot * kLuLeaf;
#pragma unroll
    for (int k = 0; k < kLuLeaf; ++k)
      if (k < count) dst[k] = vals[first + k];
  }
}

// Rows [c, n): clear the pivot flags and publish the candidates of column c.
__global__ void __launch_bounds__(kLuRows) lu_leaf_init(double* A, int64_t lda, int n, int c,
                                                        int cend, LuWork w) {
  const int i = c + (int)blockIdx.x * kLuRows + (int)threadIdx.x;
  const int nc = cend - c;
  double vals[kLuLeaf];
  double v = -1.0;
  int r = 0x7fffffff;
  if (i < n) {
    w.done[i] = 0;
#pragma unroll
    for (int k = 0; k < kLuLeaf; ++k)
      if (k < nc) vals[k] = A[i + (int64_t)(c + k) * lda];
    v = lu_mag(vals[0]);
    r = i;
  }
  lu_argmax_block(v, r);
  lu_publish(w, 0, v, r, i, vals, 0, nc);
}

// Column cj = c + j of the leaf [c, cend): choose the pivot among the
// candidates, eliminate it from every other unflagged row of the leaf, and
// publish the candidates of column cj + 1.
__global__ void __launch_bounds__(kLuRows) lu_leaf_col(double* A, int64_t lda, int n, int c,
                                                       int j, int cend, int G, LuWork w) {
  __shared__ double u[kLuLeaf];
  __shared__ int ps, gs;
  const int cj = c + j;
  const int ncol = cend - cj;                      // columns cj .. cend-1
  const int i = c + (int)blockIdx.x * kLuRows + (int)threadIdx.x;
  // independent loads first: this thread's row and flag, the candidates
  double vals[kLuLeaf];
  bool mine = false;
  if (i < n) {
    mine = !w.done[i];
#pragma unroll
    for (int k = 0; k < kLuLeaf; ++k)
      if (k < ncol) vals[k] = A[i + (int64_t)(cj + k) * lda];
  }
  const int rb = (j & 1) * w.cstride;
  if (threadIdx.x < 64) {
    double v = -1.0;
    int r = 0x7fffffff, g = 0;
    for (int t = (int)threadIdx.x; t < G; t += 64) {
      const double tv = w.candv[rb + t];
      const int tr = w.candi[rb + t];
      if (tv > v || (tv == v && tr < r)) {
        v = tv;
        r = tr;
        g = t;
      }
    }
    for (int o = 32; o >= 1; o >>= 1) {
      const double ov = __shfl_xor(v, o);
      const int orr = __shfl_xor(r, o), og = __shfl_xor(g, o);
      if (ov > v || (ov == v && orr < r)) {
        v = ov;
        r = orr;
        g = og;
      }
    }
    if (threadIdx.x == 0) {
      ps = r;
      gs = g;
    }
  }
  __syncthreads();
  // rows [cj, n) hold n - cj >= 1 unflagged rows, so the search always
  // returns one; the clamp only keeps the accesses below in bounds regardless
  const int p = ps < n ? ps : cj;
  if ((int)threadIdx.x < ncol)
    u[threadIdx.x] = w.candrow[(int64_t)(rb + gs) * kLuLeaf + threadIdx.x];
  __syncthreads();
  const double piv = u[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    w.piv[j] = p;
    if (piv == 0.0 && *w.info == 0) *w.info = cj + 1;
  }
  double v = -1.0;
  int r = 0x7fffffff;
  if (i < n && mine) {
    if (i == p) {
      w.done[i] = 1;
    } else {
      if (piv != 0.0) {
        const double l = vals[0] / piv;
        vals[0] = l;
        A[i + (int64_t)cj * lda] = l;
#pragma unroll
        for (int k = 1; k < kLuLeaf; ++k)
          if (k < ncol) {
            vals[k] = fma(-l, u[k], vals[k]);
            A[i + (int64_t)(cj + k) * lda] = vals[k];
          }
      }
      if (ncol > 1) {
        v = lu_mag(vals[1]);
        r = i;
      }
    }
  }
  if (ncol > 1) {
    lu_argmax_block(v, r);
    lu_publish(w, (j + 1) & 1, v, r, i, vals, 1, ncol - 1);
  }
}

// The leaf factored by one workgroup that holds its rows in registers: thread
// t has rows c + t + kLuWgThreads k (k < NR) of the leaf's W columns, NR x W
// <= 96 doubles.  Per column: every wave takes its own maximum (DPP), its
// winner copies its row to the wave's LDS slot, one barrier, and all waves
// pick the best slot, whose row is already the pivot row.  The slots alternate
// by column, so that barrier is the only one.  Eight waves of many rows rather
// than sixteen of few: the search and the pivot choice cost a wave the same
// whatever its rows, and two waves per SIMD already cover their latencies.
//   The column at hand is always register 0: the update of column q + 1 writes
// register q, so that one loop body serves eight columns and the code stays in
// the instruction cache.  (Every column unrolled with static register indices
// executes each instruction once a launch and is bound by fetching them.)
// Multipliers are stored in place as they are made; pivot rows are kept in LDS
// from their column on.  After the columns, wave 0 turns the pivots into
// LAPACK's interchanges and the leaf's own columns are reordered.
//   Measured: 44, 53 and 57 us a 32-column leaf of 512, 1024 and 1536 rows, 28
// to 34 us a 16-column one of 2048 to 3072, 19 to 25 us an 8-column one of 4096
// to 6144: 1.4 to 3.1 us a column, against 2.6 to 3.7 with 1024 threads and all
// columns unrolled, and 5.7 for a launch per column above 3072 rows.  Bound by the
// instructions a row takes (28 us at 6144 rows with a mask for the rows still live,
// 25 with zeros in their place), and by a column's chain of steps below that.
// Device solves: n = 2509 13.7 -> 7 ms, n = 6144 45.9 -> 26 ms.
constexpr int kLuWgThreads = 512;
constexpr int kLuWgWaves = kLuWgThreads / 64;
constexpr int kLuWgRowsMax = 12 * kLuWgThreads;  // leaf rows one workgroup takes
constexpr int kLuStage = 8;                       // columns per loop

// x of another lane of the row (or x itself where the pattern has no source)
template <int CTRL>
__device__ __forceinline__ double lu_dpp(double x) {
  const long long v = __double_as_longlong(x);
  const int lo = (int)(v & 0xffffffffLL), hi = (int)(v >> 32);
  const int l2 = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false);
  const int h2 = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)h2 << 32) | (unsigned int)l2);
}

__device__ __forceinline__ double lu_lane(double x, int lane) {
  const long long v = __double_as_longlong(x);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(v & 0xffffffffLL), lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(v >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// max without the canonicalising moves fmax adds for values from lane moves
__device__ __forceinline__ double lu_max(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// maximum over the wave (no NaN): four steps inside the 16-lane rows, two
// across them, the result read from lane 63
__device__ __forceinline__ double lu_wave_max(double v) {
  v = lu_max(v, lu_dpp<0xB1>(v));    // quad_perm [1,0,3,2]
  v = lu_max(v, lu_dpp<0x4E>(v));    // quad_perm [2,3,0,1]
  v = lu_max(v, lu_dpp<0x124>(v));   // row_ror 4
  v = lu_max(v, lu_dpp<0x128>(v));   // row_ror 8
  v = lu_max(v, lu_dpp<0x142>(v));   // row_bcast 15
  v = lu_max(v, lu_dpp<0x143>(v));   // row_bcast 31
  return lu_lane(v, 63);
}

// Pivot slots of a column: each wave's winning row (from the column on) and
// its value.
template <int W>
struct LuSlots {
  double row[2][kLuWgWaves][W];
  double mag[2][kLuWgWaves];
  int pos[2][kLuWgWaves];
};

// Up to kLuStage columns from column j0 of the leaf on, WD columns still live
// at its start (register q holds column j + q at step j).  Rows that are gone
// (pivots, bit k of `gone`, and rows past the matrix) hold zeros, which no search
// with a positive maximum picks and no update changes, so that the rows need no
// masks; a column whose maximum in a wave is zero or that holds an Inf or NaN is
// searched row by row with them.
template <int NR, int W, int WD>
__device__ __forceinline__ void lu_wg_stage(double (&vals)[NR][W], unsigned& gone, int t, int c,
                                            int j0, int nc, int n, double* A, int64_t lda,
                                            LuSlots<W>& s, double (*P)[W], int* spiv,
                                            const LuWork& w) {
  const int lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int j1 = min(j0 + kLuStage, nc);
#pragma unroll 1
  for (int j = j0; j < j1; ++j) {
    const int B = j & 1;
    int kw, lw;
    {
      double v = fabs(vals[0][0]), odd = 0.0 * vals[0][0];
      int kv = 0;
#pragma unroll
      for (int k = 1; k < NR; ++k) {
        const double x = fabs(vals[k][0]);
        kv = x > v ? k : kv;
        v = lu_max(v, x);
        odd = fma(0.0, vals[k][0], odd);
      }
      double mx = lu_wave_max(v);
      if (mx > 0.0 && !__builtin_amdgcn_ballot_w64(odd != 0.0)) {
        // the lowest row that reaches it: rows ascend with k, then with the lane
        unsigned long long m = __builtin_amdgcn_ballot_w64(v == mx);
        if (m & (m - 1)) {
          int k = 0;
          unsigned long long mk;
          while (!(mk = m & __builtin_amdgcn_ballot_w64(kv == k))) ++k;
          m = mk;
        }
        lw = __builtin_ctzll(m);
        kw = __builtin_amdgcn_readlane(kv, lw);
      } else {
        double u = -1.0;
        bool nan = false;
#pragma unroll
        for (int k = 0; k < NR; ++k) {
          const double x = vals[k][0];
          if (!(gone >> k & 1)) {
            nan |= x != x;
            u = fmax(u, fabs(x));
          }
        }
        mx = __builtin_amdgcn_ballot_w64(nan) ? (double)INFINITY : lu_wave_max(u);
        kw = -1;
        lw = 0;
#pragma unroll
        for (int k = NR - 1; k >= 0; --k) {
          const unsigned long long m =
              __builtin_amdgcn_ballot_w64(!(gone >> k & 1) && !(fabs(vals[k][0]) < mx));
          kw = m ? k : kw;
          lw = m ? __builtin_ctzll(m) : lw;
        }
      }
#pragma unroll
      for (int k = 0; k < NR; ++k)
        if (kw == k) {
          if (lane == lw) {
#pragma unroll
            for (int q = 0; q < WD; ++q) s.row[B][wv][q] = vals[k][q];
          }
        }
      if (lane == 0) {
        s.mag[B][wv] = mx;
        s.pos[B][wv] = kw < 0 ? 0x7fffffff : c + 64 * wv + lw + kLuWgThreads * kw;
      }
    }
    __syncthreads();
    const int sl = lane & (kLuWgWaves - 1);
    const double mine = s.mag[B][sl];
    const int pos = s.pos[B][sl];
    double v = lu_max(mine, lu_dpp<0xB1>(mine));
    v = lu_max(v, lu_dpp<0x4E>(v));
    v = lu_max(v, lu_dpp<0x124>(v));     // 8 slots, repeated along the row
    unsigned m = (unsigned)__builtin_amdgcn_ballot_w64(mine == v) & ((1u << kLuWgWaves) - 1);
    int g = __builtin_ctz(m);
    int p = __builtin_amdgcn_readlane(pos, g);
    for (m &= m - 1; m; m &= m - 1) {    // equal magnitudes: the lower row
      const int h = __builtin_ctz(m);
      const int q = __builtin_amdgcn_readlane(pos, h);
      if (q < p) {
        p = q;
        g = h;
      }
    }
    // the pivot row: one entry per lane, then into scalar registers (a
    // broadcast read of each would take the LDS a wave's whole return)
    const double ul = s.row[B][g][lane & (W - 1)];
    const double piv = lu_lane(ul, 0);
    if (t < WD && j + t < W) P[j][j + t] = ul;
    if (t == 0) {
      spiv[j] = p;
      if (piv == 0.0 && *w.info == 0) *w.info = c + j + 1;
    }
    if (g == wv) {                       // the pivot row is gone
#pragma unroll
      for (int k = 0; k < NR; ++k)
        if (kw == k) {
          if (lane == lw) {
            gone |= 1u << k;
#pragma unroll
            for (int q = 0; q < WD; ++q) vals[k][q] = 0.0;
          }
        }
    }
    double* a = A + (int64_t)(c + j) * lda + c + t;
    // quotients by the rounded reciprocal with one residual correction (|value| <=
    // |pivot|): the first is off by 2^-52 of itself at most, the correction's own
    // error is 2^-52 of that, so the sum before its rounding is the quotient to some
    // 2^-103 and the result is within half an ulp and a little; pivots whose
    // reciprocal could leave the normal range are divided by, and under a zero pivot
    // the column (all zeros) is left as it is
    double l[NR];
    if (__builtin_amdgcn_ballot_w64(fabs(piv) > 0x1p-1000 && fabs(piv) < 0x1p1000)) {
      const double rp = 1.0 / piv;
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        const double q = vals[k][0] * rp;
        l[k] = fma(fma(-q, piv, vals[k][0]), rp, q);
      }
    } else {
      const double by = piv == 0.0 ? 1.0 : piv;
#pragma unroll
      for (int k = 0; k < NR; ++k) l[k] = vals[k][0] / by;
    }
    // (a row that is gone stores what nothing reads; the last ones may lie past
    // the matrix)
    constexpr int kSure = NR > 6 ? NR - 2 : NR - 1;
#pragma unroll
    for (int k = 0; k < NR; ++k)
      if (k < kSure || c + t + kLuWgThreads * k < n) a[kLuWgThreads * k] = l[k];
#pragma unroll
    for (int q = 1; q < WD; ++q) {
      const double u = lu_lane(ul, q);
#pragma unroll
      for (int k = 0; k < NR; ++k) vals[k][q - 1] = fma(-l[k], u, vals[k][q]);
    }
  }
}

// LAPACK interchanges and net row movement of a leaf from its pivot rows, by
// one wavefront: at step j the row chosen (original position piv[j]) is
// swapped with whatever row is at position c + j.  Only positions touched by
// this leaf's swaps differ from the identity; they are kept as (position,
// row) pairs, one pair per lane, found by ballot.  Returns the pair of this
// lane (key -1: none).
__device__ __forceinline__ int2 lu_leaf_ipiv_wave(int c, int nc, const int* piv, int* ipiv) {
  const int lane = (int)(threadIdx.x & 63);
  int key = -1, val = -1, m = 0;
  for (int j = 0; j < nc; ++j) {
    const int want = __builtin_amdgcn_readfirstlane(piv[j]);
    const int pj = c + j;
    const unsigned long long hv = __builtin_amdgcn_ballot_w64(key >= 0 && val == want);
    const int q = hv ? __builtin_amdgcn_readlane(key, __builtin_ctzll(hv)) : want;
    const unsigned long long hp = __builtin_amdgcn_ballot_w64(key == pj);
    const int at_pj = hp ? __builtin_amdgcn_readlane(val, __builtin_ctzll(hp)) : pj;
    if (lane == 0) ipiv[pj] = q + 1;
    // position pj now holds `want`, position q the row that was at pj
    if (hp) {
      if (key == pj) val = want;
    } else {
      if (lane == m) {
        key = pj;
        val = want;
      }
      ++m;
    }
    if (q != pj) {
      const unsigned long long hq = __builtin_amdgcn_ballot_w64(key == q);
      if (hq) {
        if (key == q) val = at_pj;
      } else {
        if (lane == m) {
          key = q;
          val = at_pj;
        }
        ++m;
      }
    }
  }
  return make_int2(key, val);
}

// Leaf [c, cend) of the panel that starts at k0: see above.
template <int NR, int W>
__global__ void __launch_bounds__(kLuWgThreads) lu_leaf_wg(double* A, int64_t lda, int n, int c,
                                                           int cend, int k0, LuWork w) {
  __shared__ LuSlots<W> slots;
  __shared__ double P[W][W];      // pivot row j from column j on
  __shared__ int spiv[W];
  __shared__ int dest[W];         // where row c + i goes, or -1 for a pivot row
  const int t = threadIdx.x;
  const int nc = cend - c;
  double vals[NR][W];
  unsigned gone = 0;
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    const int r = c + t + kLuWgThreads * k;
    const bool in = r < n;
    gone |= (unsigned)!in << k;
#pragma unroll
    for (int jj = 0; jj < W; ++jj)
      vals[k][jj] = (in && jj < nc) ? A[r + (int64_t)(c + jj) * lda] : 0.0;
  }
  lu_wg_stage<NR, W, W>(vals, gone, t, c, 0, nc, n, A, lda, slots, P, spiv, w);
  if constexpr (W > kLuStage)
    lu_wg_stage<NR, W, W - kLuStage>(vals, gone, t, c, kLuStage, nc, n, A, lda, slots, P, spiv, w);
  if constexpr (W > 2 * kLuStage) {
    lu_wg_stage<NR, W, W - 2 * kLuStage>(vals, gone, t, c, 2 * kLuStage, nc, n, A, lda, slots, P,
                                         spiv, w);
    lu_wg_stage<NR, W, W - 3 * kLuStage>(vals, gone, t, c, 3 * kLuStage, nc, n, A, lda, slots, P,
                                         spiv, w);
  }
  if (t < W) dest[t] = -1;
  __syncthreads();
  if (t < 64) {
    const int2 mv = lu_leaf_ipiv_wave(c, nc, spiv, w.ipiv);
    // rows that leave [c, cend): the positions below it that changed
    if (mv.x >= cend) dest[mv.y - c] = mv.x;
  }
  __syncthreads();
  int* const mkey = w.mkey + 2 * (c - k0);
  int* const mval = w.mval + 2 * (c - k0);
  if (t < nc) {
    mkey[t] = c + t;
    mval[t] = spiv[t];
    mkey[nc + t] = dest[t];
    mval[nc + t] = c + t;
  }
  // the leaf's own columns: multipliers of the pivot rows and of the rows they
  // displace move, the pivot rows' upper part comes from LDS
  constexpr int kPer = (W * W + kLuWgThreads - 1) / kLuWgThreads;
  double up[kPer], down[kPer];
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const int i = (t + e * kLuWgThreads) % W, jj = (t + e * kLuWgThreads) / W;
    up[e] = down[e] = 0.0;
    if (i < nc && jj < nc) {
      const double* a = A + (int64_t)(c + jj) * lda;
      up[e] = jj < i ? a[spiv[i]] : P[i][jj];
      if (dest[i] >= 0) down[e] = a[c + i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const int i = (t + e * kLuWgThreads) % W, jj = (t + e * kLuWgThreads) / W;
    if (i < nc && jj < nc) {
      double* a = A + (int64_t)(c + jj) * lda;
      a[c + i] = up[e];
      if (dest[i] >= 0) a[dest[i]] = down[e];
    }
  }
}

// The panel's other columns after lu_leaf_wg, one wave for each: the leaf's row
// movement and, right of the leaf, the pivot rows' solve against its unit
// lower triangle, lane i holding row i of both.  (The update of the rows below
// it is a GEMM of its own: with a workgroup doing its columns' update too, one
// CU's bandwidth bounds it, 17-19 us against 3 + 6.)
constexpr int kLuApplyCols = 4;                   // columns (waves) per workgroup
template <int W>
__global__ void __launch_bounds__(64 * kLuApplyCols) lu_leaf_apply(double* A, int64_t lda, int c,
                                                                   int cend, int k0, int kend,
                                                                   LuWork w) {
  const int t = threadIdx.x, i = t & 63, nc = cend - c;
  // columns k0 .. c-1, then cend .. kend-1
  const int at = k0 + (int)blockIdx.x * kLuApplyCols + (t >> 6);
  const int col = at < c ? at : at + nc;
  if (col >= kend) return;
  double* a = A + (int64_t)col * lda;
  const bool on = i < nc;
  double x = 0.0, d = 0.0, l[W];
  int to = -1;
  const double* l11 = A + c + (int64_t)c * lda;
  // nc == W right of the leaf: a shorter one ends its panel
#pragma unroll
  for (int j = 0; j < W; ++j)
    l[j] = col >= cend && i < W && j < i ? l11[i + (int64_t)j * lda] : 0.0;
  if (on) {
    to = w.mkey[2 * (c - k0) + nc + i];
    x = a[w.mval[2 * (c - k0) + i]];
    d = a[c + i];
  }
  if (on && to >= 0) a[to] = d;
#pragma unroll
  for (int j = 0; j + 1 < W; ++j) x = fma(-l[j], lu_lane(x, j), x);
  if (on) a[c + i] = x;
}

// Interchanges and row movement of a leaf of the multi-workgroup path.
__global__ void __launch_bounds__(64) lu_leaf_ipiv(int c, int nc, int k0, LuWork w) {
  const int lane = (int)threadIdx.x;
  const int2 mv = lu_leaf_ipiv_wave(c, nc, w.piv, w.ipiv);
  if (lane < 2 * nc) {
    w.mkey[2 * (c - k0) + lane] = mv.x;
    w.mval[2 * (c - k0) + lane] = mv.y;
  }
}

// Apply the movement of the leaf [c, c + nc) to ncols columns from A on, one
// thread per column: the moved rows' values are all loaded, then all stored
// (the same result as the leaf's interchanges applied one after another).
__global__ void __launch_bounds__(256) lu_leaf_move(double* A, int64_t lda, int ncols, int c,
                                                    int nc, int k0, LuWork w) {
  __shared__ int sk[2 * kLuLeaf], sv[2 * kLuLeaf];
  const int t = threadIdx.x;
  if (t < 2 * kLuLeaf) {
    sk[t] = t < 2 * nc ? w.mkey[2 * (c - k0) + t] : -1;
    sv[t] = t < 2 * nc ? w.mval[2 * (c - k0) + t] : 0;
  }
  __syncthreads();
  const int col = (int)blockIdx.x * 256 + t;
  if (col >= ncols) return;
  double* a = A + (int64_t)col * lda;
  double v[2 * kLuLeaf];
#pragma unroll
  for (int k = 0; k < 2 * kLuLeaf; ++k)
    if (sk[k] >= 0) v[k] = a[sv[k]];
#pragma unroll
  for (int k = 0; k < 2 * kLuLeaf; ++k)
    if (sk[k] >= 0) a[sk[k]] = v[k];
}

// The panel's net row movement from its leaves' (columns cut[0] < cut[1] < ..
// relative to the panel, cut[nleaf] its width), over the rows [k0, n): the
// rows are replayed leaf by leaf in an LDS table, as offsets from k0.
constexpr int kLuPermRows = 65536;               // rows the table holds
constexpr int kLuMaxLeaves = kLuPanel / 8;
struct LuCuts {
  short n;
  short cut[kLuMaxLeaves + 1];
};
__global__ void __launch_bounds__(256) lu_panel_perm(int k0, int nb, int n, LuCuts cuts,
                                                     LuWork w) {
  __shared__ unsigned short pr[kLuPermRows];
  __shared__ int count;
  const int t = threadIdx.x, rows = n - k0;
  for (int i = t; i < rows; i += 256) pr[i] = (unsigned short)i;
  if (t == 0) count = nb;
  __syncthreads();
  for (int f = 0; f < cuts.n; ++f) {
    const int e0 = 2 * cuts.cut[f], e1 = 2 * cuts.cut[f + 1];   // at most 2 kLuLeaf entries
    const bool on = e0 + t < e1;
    const int key = on ? w.mkey[e0 + t] : -1;
    const unsigned short v = key >= 0 ? pr[w.mval[e0 + t] - k0] : 0;
    __syncthreads();
    if (key >= 0) pr[key - k0] = v;
    __syncthreads();
  }
  for (int i = t; i < rows; i += 256) {
    const int from = pr[i];
    if (i < nb) {
      w.pkey[i] = k0 + i;
      w.pval[i] = k0 + from;
    } else if (from != i) {
      const int e = atomicAdd(&count, 1);        // at most nb rows below the panel change
      w.pkey[e] = k0 + i;
      w.pval[e] = k0 + from;
    }
  }
  __syncthreads();
  if (t == 0) *w.pcount = count;
}

// Apply the panel's movement to the columns outside [k0, k0 + nb) and to the
// right-hand sides: kLuMoveCols columns per workgroup, a thread per entry, so
// that the panel's own rows are read and written as contiguous runs.
constexpr int kLuMoveCols = 8;
__global__ void __launch_bounds__(512) lu_panel_move(double* A, int64_t lda, int n, int k0, int nb,
                                                     double* B, int64_t ldb, int nrhs, LuWork w) {
  static_assert(2 * kLuPanel <= 512, "one thread per entry");
  const int t = threadIdx.x;
  const bool on = t < *w.pcount;
  const int key = on ? w.pkey[t] : 0, val = on ? w.pval[t] : 0;
  const bool moves = on && key != val;
  double v[kLuMoveCols];
  double* at[kLuMoveCols];
#pragma unroll
  for (int q = 0; q < kLuMoveCols; ++q) {
    const int i = (int)blockIdx.x * kLuMoveCols + q;
    at[q] = nullptr;
    if (i < n - nb) at[q] = A + (int64_t)(i < k0 ? i : i + nb) * lda;
    else if (i < n - nb + nrhs) at[q] = B + (int64_t)(i - (n - nb)) * ldb;
    if (moves && at[q]) v[q] = at[q][val];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kLuMoveCols; ++q)
    if (moves && at[q]) at[q][key] = v[q];
}

// The leaf [c, cend) of the panel [k0, kend) and its movement and solve in the
// panel's other columns; its width is lu_leaf_width(n - c).
template <int NR, int W>
void launch_leaf_wg(hipStream_t s, double* dA, int64_t lda, int n, int c, int cend, int k0,
                    int kend, const LuWork& w) {
  hipLaunchKernelGGL((lu_leaf_wg<NR, W>), dim3(1), dim3(kLuWgThreads), 0, s, dA, lda, n, c, cend,
                     k0, w);
  const int other = kend - k0 - (cend - c);
  if (other > 0)
    hipLaunchKernelGGL(lu_leaf_apply<W>, dim3((other + kLuApplyCols - 1) / kLuApplyCols),
                       dim3(64 * kLuApplyCols), 0, s, dA, lda, c, cend, k0, kend, w);
}

void launch_leaf(hipStream_t s, double* dA, int64_t lda, int n, int c, int cend, int k0, int kend,
                 const LuWork& w) {
#define PSX_LEAF(NR, W) launch_leaf_wg<NR, W>(s, dA, lda, n, c, cend, k0, kend, w)
  switch ((n - c + kLuWgThreads - 1) / kLuWgThreads) {
    case 1: return PSX_LEAF(1, 32);
    case 2: return PSX_LEAF(2, 32);
    case 3: return PSX_LEAF(3, 32);
    case 4: return PSX_LEAF(4, 16);
    case 5: return PSX_LEAF(5, 16);
    case 6: return PSX_LEAF(6, 16);
    case 7:
    case 8: return PSX_LEAF(8, 8);
    case 9:
    case 10: return PSX_LEAF(10, 8);
    default: return PSX_LEAF(12, 8);
  }
#undef PSX_LEAF
}

// Columns of the leaf that starts with `rows` rows to factor.
int lu_leaf_width(int rows) {
  const int nr = (rows + kLuWgThreads - 1) / kLuWgThreads;
  return nr > 12 ? kLuLeaf : nr > 6 ? 8 : nr > 3 ? 16 : 32;
}
// Where an LU runs: a stream, the rocBLAS handle bound to it and a device work
// area of lu_work_bytes(n) bytes (pivot candidates, flags, the leaf's row
// movement).  Factorizations on different lanes may run at the same time.
struct LuLane {
  hipStream_t s;
  rocblas_handle h;
  void* work;
};

size_t lu_work_bytes(int n) {
  const int Gmax = (n + kLuRows - 1) / kLuRows;
  const size_t rows_bytes = 2 * (size_t)Gmax * kLuLeaf * sizeof(double);
  const size_t move_off = (rows_bytes + 24 * (size_t)Gmax + 4 * kLuLeaf + (size_t)n + 255) &
                          ~size_t(255);
  return move_off + sizeof(int) * (8 * kLuPanel + 1) + 256;
}

// ---- triangular solves with many right-hand sides ---------------------------
// Blocked left substitution X = T^{-1} B for the LU factors (T = unit lower L
// or upper U) and m right-hand sides, in kTsmRows-row blocks: the diagonal
// block is solved by substitution (trsm_block), and the rows still to come are
// updated by a rocBLAS GEMM of depth kTsmRows.  Substitution keeps LAPACK's
// backward error on ill-conditioned U, which a trsm built on inverted diagonal
// blocks does not.
//   A wave takes kTsmCols right-hand sides, lane i holding rows i, i + 64, ..
// of the block; the value solved at a step goes through scalar registers to
// all lanes.  The triangle passes through LDS, kTsmAhead columns at a time,
// one set ahead of the steps, so that a workgroup's waves read it from L2
// once: with each wave reading it for itself the L2 bounds the kernel (103 and
// 169 us at m = 2509; 34 and 58 us with LDS).  Issue-bound on the broadcasts,
// the quotients and the updates.  64-row blocks, one right-hand side a thread,
// ran 45 us each (180 for 256 rows) on 14 workgroups, and their depth-64 GEMMs
// were bound by the traffic of B.
constexpr int kTsmRows = 256;
constexpr int kTsmCols = 2;
constexpr int kTsmWaves = 8;
constexpr int kTsmAhead = 16;

// ROWS: rows the diagonal block has at most.
template <bool UPPER, int ROWS>
__global__ void __launch_bounds__(64 * kTsmWaves) trsm_block(const double* __restrict__ A,
                                                             int64_t lda, int n, int R0,
                                                             double* __restrict__ B, int64_t ldb,
                                                             int m) {
  constexpr int kTsmSub = ROWS / 64;
  constexpr int kTsmStage = kTsmAhead * ROWS / (64 * kTsmWaves);  // values a thread stages
  __shared__ double Ts[2][kTsmAhead][ROWS];
  const int t = threadIdx.x, lane = t & 63;
  const int col0 = __builtin_amdgcn_readfirstlane(
      ((int)blockIdx.x * kTsmWaves + (t >> 6)) * kTsmCols);
  const int cn = min(ROWS, n - R0);
  const double* T = A + R0 + (int64_t)R0 * lda;     // T[row + column lda]
  double* b = B + R0 + (int64_t)col0 * ldb;
  // acc: what the sub-blocks already solved take from one still to come,
  // summed by itself and subtracted once, as the GEMM between blocks does
  double x[kTsmSub][kTsmCols], acc[kTsmSub][kTsmCols], d[kTsmSub], rd[kTsmSub];
  bool plain = true;
#pragma unroll
  for (int s = 0; s < kTsmSub; ++s) {
    const int r = 64 * s + lane;
#pragma unroll
    for (int q = 0; q < kTsmCols; ++q) {
      x[s][q] = r < cn && col0 + q < m ? b[r + (int64_t)q * ldb] : 0.0;
      acc[s][q] = 0.0;
    }
    d[s] = UPPER && r < cn ? T[r + (int64_t)r * lda] : 1.0;
    rd[s] = 1.0 / d[s];
    plain &= fabs(d[s]) > 0x1p-1000 && fabs(d[s]) < 0x1p1000;
  }
  // every pivot's reciprocal in the normal range: quotients by it, with one
  // residual correction (good to half an ulp and a little, as in lu_wg_stage)
  const bool fast = __builtin_amdgcn_ballot_w64(!plain) == 0;
  // sets of kTsmAhead columns, from the first (lower) or last (upper) that
  // holds one of the block; a thread stages kTsmStage of a set's entries in
  // its row, zero beyond the block
  const int row = t % ROWS, part = (t / ROWS) * kTsmStage;
  double ahead[kTsmStage];
  auto load = [&](int f) {
#pragma unroll
    for (int e = 0; e < kTsmStage; ++e) {
      const int j = f * kTsmAhead + part + e;
      ahead[e] = row < cn && j < cn ? T[row + (int64_t)j * lda] : 0.0;
    }
  };
  constexpr int kSets = 64 / kTsmAhead;             // of a 64-row sub-block
  const int last = (cn - 1) / kTsmAhead;
  load(UPPER ? last : 0);
#pragma unroll
  for (int ss = 0; ss < kTsmSub; ++ss) {
    const int s = UPPER ? kTsmSub - 1 - ss : ss;
    const int f0 = s * kSets, f1 = min(f0 + kSets - 1, last);
#pragma unroll
    for (int c = 0; c < kTsmCols; ++c) x[s][c] -= acc[s][c];
#pragma unroll 1
    for (int i = f0; i <= f1; ++i) {
      const int f = UPPER ? f1 - (i - f0) : i, buf = f & 1;
#pragma unroll
      for (int e = 0; e < kTsmStage; ++e) Ts[buf][part + e][row] = ahead[e];
      __syncthreads();                              // also ends the reads of set f -+ 1
      const int nf = UPPER ? f - 1 : f + 1;
      if (nf >= 0 && nf <= last) load(nf);
      const int j0 = (f - f0) * kTsmAhead;
#pragma unroll
      for (int u = 0; u < kTsmAhead; ++u) {
        const int e = UPPER ? kTsmAhead - 1 - u : u, j = j0 + e;
        const bool off = UPPER ? lane < j : lane > j;
        double tv[kTsmSub];
#pragma unroll
        for (int q = 0; q < kTsmSub; ++q)
          if (UPPER ? q <= s : q >= s) tv[q] = Ts[buf][e][64 * q + lane];
#pragma unroll
        for (int c = 0; c < kTsmCols; ++c) {
          double y = x[s][c], xj;
          if (UPPER) {
            if (fast) {
              const double z = y * rd[s];
              const double w = fma(fma(-z, d[s], y), rd[s], z);
              xj = lu_lane(w, j);
              // an overflow, whose correction is NaN, or a NaN: divide
              if ((__double2hiint(xj) & 0x7ff00000) != 0x7ff00000) {
                y = w;
              } else {
                y = y / d[s];
                xj = lu_lane(y, j);
              }
            } else {
              y = y / d[s];
              xj = lu_lane(y, j);
            }
          } else {
            xj = lu_lane(y, j);
          }
          const double own = fma(-tv[s], xj, x[s][c]);
          x[s][c] = off ? own : (UPPER && lane == j) ? y : x[s][c];
#pragma unroll
          for (int q = 0; q < kTsmSub; ++q)
            if (UPPER ? q < s : q > s) acc[q][c] = fma(tv[q], xj, acc[q][c]);
        }
      }
    }
  }
#pragma unroll
  for (int s = 0; s < kTsmSub; ++s) {
    const int r = 64 * s + lane;
#pragma unroll
    for (int q = 0; q < kTsmCols; ++q)
      if (r < cn && col0 + q < m) b[r + (int64_t)q * ldb] = x[s][q];
  }
}

static unsigned trsm_grid(int m) {
  return (unsigned)((m + kTsmWaves * kTsmCols - 1) / (kTsmWaves * kTsmCols));
}

// U rows of the factorization: B (nb x m) = L^{-1} B with the unit lower nb x nb
// block at A, nb <= ROWS, in the same matrix.  (rocBLAS's trsm inverts diagonal
// blocks and multiplies in several launches: 85 us at nb = 128, m = 2400 to 6000.)
template <int ROWS>
static void panel_trsm(hipStream_t s, int nb, const double* A, int64_t lda, double* B, int m) {
  hipLaunchKernelGGL((trsm_block<false, ROWS>), dim3(trsm_grid(m)), dim3(64 * kTsmWaves), 0, s, A,
                     lda, nb, 0, B, lda, m);
  PSX_HIP(hipGetLastError());
}

// dA (n x n) becomes its LU factors; the interchanges are applied to the nrhs
// columns of dB on the way.
void lu_factor_on(const LuLane& L, int n, double* dA, int64_t lda, int* dipiv, int* dinfo,
                  double* dB = nullptr, int64_t ldb = 0, int nrhs = 0) {
  rocblas_handle h = L.h;
  hipStream_t s = L.s;
  const int Gmax = (n + kLuRows - 1) / kLuRows;
  const size_t rows_bytes = 2 * (size_t)Gmax * kLuLeaf * sizeof(double);
  const size_t move_off = (rows_bytes + 24 * (size_t)Gmax + 4 * kLuLeaf + (size_t)n + 255) &
                          ~size_t(255);
  char* base = (char*)L.work;
  LuWork w;
  w.cstride = Gmax;
  w.candrow = (double*)base;                                  // 2 Gmax kLuLeaf doubles
  w.candv = (double*)(base + rows_bytes);                     // 2 Gmax doubles
  w.candi = (int*)(base + rows_bytes + 16 * (size_t)Gmax);    // 2 Gmax ints
  w.piv = (int*)(base + rows_bytes + 24 * (size_t)Gmax);      // kLuLeaf ints
  w.done = (unsigned char*)(base + rows_bytes + 24 * (size_t)Gmax + 4 * kLuLeaf);  // n flags
  w.mkey = (int*)(base + move_off);                           // 2 kLuPanel ints each
  w.mval = w.mkey + 2 * kLuPanel;
  w.pkey = w.mval + 2 * kLuPanel;
  w.pval = w.pkey + 2 * kLuPanel;
  w.pcount = w.pval + 2 * kLuPanel;                           // 1 int
  w.ipiv = dipiv;
  w.info = dinfo;
  PSX_HIP(hipMemsetAsync(dinfo, 0, sizeof(int), s));
  const double one = 1.0, mone = -1.0;
  for (int k = 0; k < n; k += kLuPanel) {
    const int kend = std::min(n, k + kLuPanel), nb = kend - k;
    // the panel's net movement is replayed in LDS, which bounds its rows
    const bool deferred = n - k <= kLuPermRows;
    LuCuts cuts{};
    for (int cl = k; cl < kend;) {
      const int rows = n - cl;
      const bool one_wg = rows <= kLuWgRowsMax;
      const int cend = std::min(kend, cl + lu_leaf_width(rows));
      const int nc = cend - cl;
      if (one_wg) {
        launch_leaf(s, dA, lda, n, cl, cend, k, kend, w);
      } else {
        const int G = (rows + kLuRows - 1) / kLuRows;
        hipLaunchKernelGGL(lu_leaf_init, dim3(G), dim3(kLuRows), 0, s, dA, lda, n, cl, cend, w);
        for (int j = 0; j < nc; ++j)
          hipLaunchKernelGGL(lu_leaf_col, dim3(G), dim3(kLuRows), 0, s, dA, lda, n, cl, j, cend,
                             G, w);
        hipLaunchKernelGGL(lu_leaf_ipiv, dim3(1), dim3(64), 0, s, cl, nc, k, w);
        hipLaunchKernelGGL(lu_leaf_move, dim3((nb + 255) / 256), dim3(256), 0, s,
                           dA + (int64_t)k * lda, lda, nb, cl, nc, k, w);
        if (cend < kend)   // rest of the panel: U = L11^-1 A
          panel_trsm<64>(s, nc, dA + cl + (int64_t)cl * lda, lda, dA + cl + (int64_t)cend * lda,
                         kend - cend);
      }
      if (!deferred) {
        if (k > 0)
          hipLaunchKernelGGL(lu_leaf_move, dim3((k + 255) / 256), dim3(256), 0, s, dA, lda, k, cl,
                             nc, k, w);
        if (kend < n)
          hipLaunchKernelGGL(lu_leaf_move, dim3((n - kend + 255) / 256), dim3(256), 0, s,
                             dA + (int64_t)kend * lda, lda, n - kend, cl, nc, k, w);
        if (nrhs > 0)
          hipLaunchKernelGGL(lu_leaf_move, dim3((nrhs + 255) / 256), dim3(256), 0, s, dB, ldb,
                             nrhs, cl, nc, k, w);
      }
      PSX_HIP(hipGetLastError());
      if (cend < kend)     // the rows below it
        PSX_ROC(rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, n - cend,
                              kend - cend, nc, &mone, dA + cend + (int64_t)cl * lda,
                              (rocblas_int)lda, dA + cl + (int64_t)cend * lda, (rocblas_int)lda,
                              &one, dA + cend + (int64_t)cend * lda, (rocblas_int)lda));
      cuts.cut[cuts.n++] = (short)(cl - k);
      cl = cend;
    }
    cuts.cut[cuts.n] = (short)nb;
    const int others = n - nb + nrhs;
    if (deferred && others > 0) {
      hipLaunchKernelGGL(lu_panel_perm, dim3(1), dim3(256), 0, s, k, nb, n, cuts, w);
      hipLaunchKernelGGL(lu_panel_move, dim3((others + kLuMoveCols - 1) / kLuMoveCols), dim3(512),
                         0, s, dA, lda, n, k, nb, dB, ldb, nrhs, w);
      PSX_HIP(hipGetLastError());
    }
    if (kend < n) {        // trailing matrix
      double* L11 = dA + k + (int64_t)k * lda;
      double* A12 = dA + k + (int64_t)kend * lda;
      panel_trsm<kLuPanel>(s, nb, L11, lda, A12, n - kend);
      PSX_ROC(rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, n - kend, n - kend,
                            nb, &mone, dA + kend + (int64_t)k * lda, (rocblas_int)lda, A12,
                            (rocblas_int)lda, &one, dA + kend + (int64_t)kend * lda,
                            (rocblas_int)lda));
    }
  }
}

void lu_factor_dev(Ctx* c, int n, double* dA, int64_t lda, int* dipiv, int* dinfo) {
  lu_factor_on(LuLane{c->stream, blas(c), ctx_scratch(c, lu_work_bytes(n))}, n, dA, lda, dipiv,
               dinfo);
}

// ---- triangular solves with the LU factors, one right-hand side ------------
// A blocked substitution in kTrsRows-row blocks, one launch per block step.
// Forward (unit lower L): launch k updates every row block from k on with the
// solution of block k-1, then workgroup 0, which holds block k, solves block
// k's diagonal triangle.  Back (U, diagonal included): launch k, from the last
// block down, updates row blocks k, k-1, .., 0 with block k+1's solution, and
// workgroup 0 solves block k.  Each launch reads its columns once, so a
// triangle costs n^2/2 reads.
//   The update is a column-major GEMV with two threads per row, each taking
// 64 columns with all its loads in flight.  Workgroup 0 stages the whole
// diagonal block in LDS (132 KB) while it runs its own rows' update, then
// solves the block from LDS in two 64-row sub-blocks, one wave each, the
// solved value broadcast by v_readlane.
constexpr int kTrsRows = 128;
constexpr int kTrsLd = kTrsRows + 1;   // LDS column stride of the diagonal block
constexpr int kTrsMaxRhs = 4;          // more right-hand sides take the blocked trsm below

// lane j's value in every lane (j uniform: two v_readlane_b32)
__device__ inline double trs_bcast(double v, int j) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, j);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), j);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <bool UPPER>
__global__ void __launch_bounds__(256) trs_step(const double* __restrict__ A, int64_t lda, int n,
                                                int k, double* __restrict__ x) {
  __shared__ double D[kTrsRows * kTrsLd];  // diagonal block, column-major (workgroup 0)
  __shared__ double xs[kTrsRows];          // source block's solution
  __shared__ double part[2][kTrsRows];     // the two half-row partial sums
  const int nb = (n + kTrsRows - 1) / kTrsRows;
  const int t = threadIdx.x;
  const int rl = t & (kTrsRows - 1), h = t >> 7;  // row in the block, column half
  const int rb = UPPER ? k - (int)blockIdx.x : k + (int)blockIdx.x;
  const int R0 = rb * kTrsRows;
  const int r = R0 + rl;
  const bool diag = blockIdx.x == 0;
  const int cn = min(kTrsRows, n - R0);  // rows in this block (= columns of the diagonal)
  if (diag) {
    // thread t fills row t & 127 of columns 2m + (t >> 7), m = 0..63, 32 loads
    // in flight at a time
    const bool rin = rl < cn;
    const double* a = A + (R0 + (rin ? rl : 0)) + (int64_t)R0 * lda;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      double v[32];
#pragma unroll
      for (int q = 0; q < 32; ++q) {
        const int ic = 2 * (half * 32 + q) + h;
        v[q] = (rin && ic < cn) ? a[(int64_t)ic * lda] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < 32; ++q) D[(2 * (half * 32 + q) + h) * kTrsLd + rl] = v[q];
    }
  }
  double y = (h == 0 && r < n) ? x[r] : 0.0;
  const int src = UPPER ? k + 1 : k - 1;
  if (src >= 0 && src < nb) {
    const int c0 = src * kTrsRows, sn = min(kTrsRows, n - c0);
    if (t < sn) xs[t] = x[c0 + t];
    __syncthreads();
    double p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0;
    if (r < n) {
      const int j0 = h * 64;
      const double* a = A + r + (int64_t)(c0 + j0) * lda;
      if (sn == kTrsRows) {  // a full source block: all 64 loads in flight
        double v[64];
#pragma unroll
        for (int q = 0; q < 64; ++q) v[q] = a[(int64_t)q * lda];
#pragma unroll
        for (int q = 0; q < 64; q += 4) {
          p0 = fma(v[q], xs[j0 + q], p0);
          p1 = fma(v[q + 1], xs[j0 + q + 1], p1);
          p2 = fma(v[q + 2], xs[j0 + q + 2], p2);
          p3 = fma(v[q + 3], xs[j0 + q + 3], p3);
        }
      } else {
        const int m = min(sn, j0 + 64) - j0;
        for (int q = 0; q < m; ++q) p0 = fma(a[(int64_t)q * lda], xs[j0 + q], p0);
      }
    }
    part[h][rl] = (p0 + p1) + (p2 + p3);
    __syncthreads();
    if (h == 0) y -= part[0][rl] + part[1][rl];
  }
  if (!diag) {
    if (h == 0 && r < n) x[r] = y;
    return;
  }
  __syncthreads();  // D complete
  // the diagonal block: rows 0..63 are wave 0, rows 64..127 wave 1
  const int w = t >> 6, lane = t & 63;
  const int nsub = (cn + 63) >> 6;
  for (int q = 0; q < nsub; ++q) {
    const int s = UPPER ? nsub - 1 - q : q;
    const int s0 = s * 64, sn = min(64, cn - s0);
    if (w == s) {
      const double* d = D + s0 * kTrsLd + s0 + lane;  // column j at d[j * kTrsLd]
      double T[64];
#pragma unroll
      for (int j = 0; j < 64; ++j) T[j] = d[j * kTrsLd];
      if (!UPPER) {
#pragma unroll
        for (int j = 0; j < 64; ++j) {
          if (j < sn) {
            const double xj = trs_bcast(y, j);
            if (lane > j) y = fma(-T[j], xj, y);
          }
        }
      } else {
#pragma unroll
        for (int j = 63; j >= 0; --j) {
          if (j < sn) {
            if (lane == j) y = y / T[j];
            const double xj = trs_bcast(y, j);
            if (lane < j) y = fma(-T[j], xj, y);
          }
        }
      }
      if (lane < sn) xs[s0 + lane] = y;
    }
    __syncthreads();
    const bool later = t < cn && (UPPER ? (w < s) : (w > s));
    if (later) {
      const double* d = D + s0 * kTrsLd + t;
      double p0 = 0.0, p1 = 0.0;
      int j = 0;
      for (; j + 2 <= sn; j += 2) {
        p0 = fma(d[j * kTrsLd], xs[s0 + j], p0);
        p1 = fma(d[(j + 1) * kTrsLd], xs[s0 + j + 1], p1);
      }
      if (j < sn) p0 = fma(d[j * kTrsLd], xs[s0 + j], p0);
      y -= p0 + p1;
    }
  }
  if (t < cn) x[r] = y;
}

// x = L^{-1} x, then x = U^{-1} x, with the packed LU factors of dA, on stream s.
void lu_trs_on(hipStream_t s, int n, const double* dA, int64_t lda, double* dx) {
  const int nb = (n + kTrsRows - 1) / kTrsRows;
  // (the first step of each sweep has no source block: only the diagonal)
  for (int k = 0; k < nb; ++k)
    hipLaunchKernelGGL(trs_step<false>, dim3(k == 0 ? 1 : nb - k), dim3(256), 0, s, dA, lda, n,
                       k, dx);
  for (int k = nb - 1; k >= 0; --k)
    hipLaunchKernelGGL(trs_step<true>, dim3(k == nb - 1 ? 1 : k + 1), dim3(256), 0, s, dA, lda,
                       n, k, dx);
  PSX_HIP(hipGetLastError());
}

void lu_trs_dev(Ctx* c, int n, const double* dA, int64_t lda, double* dx) {
  lu_trs_on(c->stream, n, dA, lda, dx);
}

// B (n x m, ldb) = T^{-1} B with T the unit lower (UPPER false) or upper
// factor packed in dA.
static void trsm_left_dev(Ctx* c, bool upper, int n, const double* dA, int64_t lda, double* dB,
                          int64_t ldb, int m) {
  rocblas_handle h = blas(c);
  hipStream_t s = c->stream;
  const int nb = (n + kTsmRows - 1) / kTsmRows;
  const unsigned g = trsm_grid(m);
  const double one = 1.0, mone = -1.0;
  for (int q = 0; q < nb; ++q) {
    const int R0 = (upper ? nb - 1 - q : q) * kTsmRows, cn = std::min(kTsmRows, n - R0);
    if (upper)
      hipLaunchKernelGGL((trsm_block<true, kTsmRows>), dim3(g), dim3(64 * kTsmWaves), 0, s, dA, lda, n, R0, dB,
                         ldb, m);
    else
      hipLaunchKernelGGL((trsm_block<false, kTsmRows>), dim3(g), dim3(64 * kTsmWaves), 0, s, dA, lda, n, R0, dB,
                         ldb, m);
    PSX_HIP(hipGetLastError());
    if (!upper && R0 + cn < n)  // rows below: B2 -= L21 X1
      PSX_ROC(rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, n - R0 - cn, m, cn,
                            &mone, dA + (R0 + cn) + (int64_t)R0 * lda, (rocblas_int)lda,
                            dB + R0, (rocblas_int)ldb, &one, dB + R0 + cn, (rocblas_int)ldb));
    if (upper && R0 > 0)        // rows above: B0 -= U01 X1
      PSX_ROC(rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, R0, m, cn, &mone,
                            dA + (int64_t)R0 * lda, (rocblas_int)lda, dB + R0, (rocblas_int)ldb,
                            &one, dB, (rocblas_int)ldb));
  }
}

// The row order LAPACK's interchanges produce, perm[i] = the original row
// that ends at position i, built by one thread in LDS (the interchanges are
// sequential by definition) and written out by the workgroup.
constexpr int kPermMax = 16384;
__global__ void __launch_bounds__(256) lu_perm(const int* __restrict__ ipiv, int n,
                                               int* __restrict__ perm) {
  __shared__ int pr[kPermMax], iv[kPermMax];
  for (int i = threadIdx.x; i < n; i += 256) {
    pr[i] = i;
    iv[i] = ipiv[i] - 1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 0; i < n; ++i) {
      const int q = iv[i];
      if (q != i && q > i && q < n) {
        const int t = pr[i];
        pr[i] = pr[q];
        pr[q] = t;
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 256) perm[i] = pr[i];
}

// Column blockIdx.x of B (n rows, ldb) reordered in place: b[i] = b[perm[i]],
// through LDS.
__global__ void __launch_bounds__(256) lu_permute_cols(const int* __restrict__ perm, int n,
                                                       double* __restrict__ B, int64_t ldb) {
  __shared__ double col[kPermMax];
  double* b = B + (int64_t)blockIdx.x * ldb;
  for (int i = threadIdx.x; i < n; i += 256) col[i] = b[i];
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += 256) b[i] = col[perm[i]];
}

// The row order of B before LAPACK's interchanges, one thread per column (after a
// zero pivot only).
__global__ void __launch_bounds__(64) lu_undo_swaps(const int* __restrict__ ipiv, int n,
                                                    double* __restrict__ B, int64_t ldb,
                                                    int nrhs) {
  const int col = (int)(blockIdx.x * 64 + threadIdx.x);
  if (col >= nrhs) return;
  double* b = B + (int64_t)col * ldb;
  for (int i = n - 1; i >= 0; --i) {
    const int q = ipiv[i] - 1;
    if (q > i && q < n) {
      const double t = b[i];
      b[i] = b[q];
      b[q] = t;
    }
  }
}

// A device array for LAPACK's interchanges: n entries, the info slot at n + 32.
static size_t pivot_bytes(int n) {
  return (sizeof(int) * ((size_t)n + 64) + 255) & ~size_t(255);
}

// SingularException for a zero pivot in a finished factorisation; waits for
// the context stream.
static void check_pivots(Ctx* c, int n, const int* ipiv) {
  ensure_stage(c);
  PSX_HIP(hipMemcpyAsync(c->flag, ipiv + n + 32, sizeof(int), hipMemcpyDeviceToHost, c->stream));
  PSX_HIP(hipStreamSynchronize(c->stream));
  PSX_REQUIRE(*c->flag == 0, PSX_ERR_SINGULAR,
              "LU: zero pivot at position " + std::to_string(*c->flag) +
                  " (Julia SingularException)");
}

// dA (n x n, lda) becomes its LU factors, dB (n x nrhs) A^{-1} dB.  With keep_b a
// singular matrix leaves dB as it was: the pivots are looked at before the
// substitution (a wait, which callers with a copy of their own do without) and the
// rows moved with the panels go back.
void lu_solve_dev(Ctx* c, int n, double* dA, int64_t lda, double* dB, int64_t ldb,
                  int nrhs, bool keep_b) {
  const size_t wb = (lu_work_bytes(n) + 255) & ~size_t(255);
  char* work = (char*)ctx_scratch(c, wb + pivot_bytes(n));
  int* ipiv = (int*)(work + wb);
  lu_factor_on(LuLane{c->stream, blas(c), work}, n, dA, lda, ipiv, ipiv + n + 32, dB, ldb, nrhs);
  if (keep_b) {
    try {
      check_pivots(c, n, ipiv);
    } catch (const Error& e) {
      if (e.code == PSX_ERR_SINGULAR && nrhs > 0) {
        hipLaunchKernelGGL(lu_undo_swaps, dim3((unsigned)((nrhs + 63) / 64)), dim3(64), 0,
                           c->stream, (const int*)ipiv, n, dB, ldb, nrhs);
        (void)hipStreamSynchronize(c->stream);
      }
      throw;
    }
  }
  if (nrhs <= kTrsMaxRhs) {
    for (int j = 0; j < nrhs; ++j) lu_trs_dev(c, n, dA, lda, dB + (int64_t)j * ldb);
  } else {
    trsm_left_dev(c, false, n, dA, lda, dB, ldb, nrhs);
    trsm_left_dev(c, true, n, dA, lda, dB, ldb, nrhs);
  }
  if (keep_b) PSX_HIP(hipStreamSynchronize(c->stream));
  else check_pivots(c, n, ipiv);
}

// Independent systems side by side.  System i runs on lane i: lane 0 is the
// context stream, lanes 1.. the context's extra streams, each with its own
// rocBLAS handle and its own part of the scratch.  The lanes start after the
// work already queued on the context stream, and the context stream waits
// for all of them, so the call keeps stream order for its caller.  The
// factorizations are latency-bound (a leaf column runs on one or a few
// workgroups), so running them at once overlaps their latencies.
void ensure_lanes(Ctx* c, int nextra) {
  for (int i = 0; i < nextra; ++i) {
    if (c->lstream[i]) continue;
    PSX_HIP(hipStreamCreateWithFlags(&c->lstream[i], hipStreamNonBlocking));
    rocblas_handle h;
    PSX_REQUIRE(rocblas_create_handle(&h) == rocblas_status_success, PSX_ERR_DEVICE,
                "rocblas_create_handle failed");
    rocblas_set_stream(h, c->lstream[i]);
    c->lblas[i] = h;
  }
  for (hipEvent_t& e : c->lane_ev)
    if (!e) PSX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
}

void lu_solve_concurrent(Ctx* c, const LuSystem* sys, int count) {
  PSX_REQUIRE(count >= 1 && count <= 1 + kLuExtraLanes, PSX_ERR_ARGUMENT,
              "too many concurrent systems");
  ensure_lanes(c, count - 1);
  std::vector<size_t> off(count + 1, 0);
  for (int i = 0; i < count; ++i) {
    PSX_REQUIRE(sys[i].nrhs >= 1 && sys[i].nrhs <= kTrsMaxRhs, PSX_ERR_ARGUMENT,
                "concurrent systems take 1 to 4 right-hand sides");
    off[i + 1] = off[i] + ((lu_work_bytes(sys[i].n) + 255) & ~size_t(255));
  }
  char* work = (char*)ctx_scratch(c, off[count]);
  blas(c);
  PSX_HIP(hipEventRecord(c->lane_ev[0], c->stream));
  try {
    for (int i = 0; i < count; ++i) {
      const LuSystem& q = sys[i];
      const LuLane L = i == 0 ? LuLane{c->stream, blas(c), work}
                              : LuLane{c->lstream[i - 1], (rocblas_handle)c->lblas[i - 1],
                                       work + off[i]};
      if (i > 0) PSX_HIP(hipStreamWaitEvent(L.s, c->lane_ev[0], 0));
      lu_factor_on(L, q.n, q.dA, q.lda, q.ipiv, q.ipiv + q.n + 32, q.dB, q.ldb, q.nrhs);
      for (int j = 0; j < q.nrhs; ++j)
        lu_trs_on(L.s, q.n, q.dA, q.lda, q.dB + (int64_t)j * q.ldb);
      PSX_HIP(hipGetLastError());
      if (i > 0) {
        PSX_HIP(hipEventRecord(c->lane_ev[i], L.s));
        PSX_HIP(hipStreamWaitEvent(c->stream, c->lane_ev[i], 0));
      }
    }
  } catch (...) {
    // nothing may still run on the caller's buffers once the error is out
    for (int i = 0; i + 1 < count; ++i) (void)hipStreamSynchronize(c->lstream[i]);
    (void)hipStreamSynchronize(c->stream);
    throw;
  }
  // SingularException for the first system with a zero pivot
  static_assert(1 + kLuExtraLanes <= kFlags, "a pinned word for each system");
  ensure_stage(c);
  int* const info = c->flag;
  for (int i = 0; i < count; ++i)
    PSX_HIP(hipMemcpyAsync(&info[i], sys[i].ipiv + sys[i].n + 32, sizeof(int),
                           hipMemcpyDeviceToHost, c->stream));
  PSX_HIP(hipStreamSynchronize(c->stream));
  for (int i = 0; i < count; ++i)
    PSX_REQUIRE(info[i] == 0, PSX_ERR_SINGULAR,
                "LU: zero pivot at position " + std::to_string(info[i]) + " of system " +
                    std::to_string(i) + " (Julia SingularException)");
}

void release_lanes(Ctx* c) {
  for (int i = 0; i < kLuExtraLanes; ++i) {
    if (c->lstream[i]) (void)hipStreamSynchronize(c->lstream[i]);
    if (c->lblas[i]) rocblas_destroy_handle(static_cast<rocblas_handle>(c->lblas[i]));
    if (c->lstream[i]) (void)hipStreamDestroy(c->lstream[i]);
    c->lblas[i] = nullptr;
    c->lstream[i] = nullptr;
  }
  for (hipEvent_t& e : c->lane_ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

// B[r0 + i, j] = -B[r0 + i, j] for i < nr, j < gridDim.y
__global__ void __launch_bounds__(256) negate_rows(double* __restrict__ B, int64_t ldb, int r0,
                                                   int nr) {
  const int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
  if (i < nr) {
    double* p = B + (int64_t)blockIdx.y * ldb + r0 + i;
    *p = -*p;
  }
}

static void transpose(Ctx* c, int n, const double* dIn, double* dOut) {
  const double one = 1.0, zero = 0.0;
  PSX_ROC(rocblas_dgeam(blas(c), rocblas_operation_transpose, rocblas_operation_none, n, n,
                        &one, dIn, n, &zero, dOut, n, dOut, n));
}

// dY = B1^{-1} Y B2^{-T}, with dT scratch of the same size; dB1, dB2 are
// overwritten by their LU factors.  dB2 == dB1 (one matrix on both sides) is
// factored once; otherwise B2 is factored on a stream of its own, beside B1's
// factorisation and solve (both are bound by the latency of one workgroup's
// leaves), once `b2` has put it on the device.
void decouple_dev(Ctx* c, int n, double* dY, double* dB1, double* dB2, double* dT,
                  const std::function<void()>& b2) {
  const bool same = dB2 == dB1;
  ensure_lanes(c, 1);
  const size_t wb = (lu_work_bytes(n) + 255) & ~size_t(255), pb = pivot_bytes(n);
  char* work = (char*)ctx_scratch(c, 2 * wb + 3 * pb);
  int* const p1 = (int*)(work + 2 * wb);
  int* const p2 = (int*)(work + 2 * wb + pb);
  int* const perm = (int*)(work + 2 * wb + 2 * pb);
  const LuLane L1{c->stream, blas(c), work};
  const LuLane L2 = same ? L1 : LuLane{c->lstream[0], (rocblas_handle)c->lblas[0], work + wb};
  const int* ip2 = same ? p1 : p2;
  PSX_HIP(hipEventRecord(c->lane_ev[0], c->stream));
  try {
    lu_factor_on(L1, n, dB1, n, p1, p1 + n + 32, dY, n, n);
    trsm_left_dev(c, false, n, dB1, n, dY, n, n);   // dY = B1^{-1} Y
    trsm_left_dev(c, true, n, dB1, n, dY, n, n);
    transpose(c, n, dY, dT);                        // dT = dY^T
    if (!same) {
      b2();
      PSX_HIP(hipStreamWaitEvent(L2.s, c->lane_ev[0], 0));
      lu_factor_on(L2, n, dB2, n, p2, p2 + n + 32);
    }
    if (n <= kPermMax)
      hipLaunchKernelGGL(lu_perm, dim3(1), dim3(256), 0, L2.s, ip2, n, perm);
    PSX_HIP(hipGetLastError());
    if (!same) {
      PSX_HIP(hipEventRecord(c->lane_ev[1], L2.s));
      PSX_HIP(hipStreamWaitEvent(c->stream, c->lane_ev[1], 0));
    }
    if (n <= kPermMax)
      hipLaunchKernelGGL(lu_permute_cols, dim3((unsigned)n), dim3(256), 0, c->stream,
                         (const int*)perm, n, dT, (int64_t)n);
    else
      PSX_ROC(rocsolver_dlaswp(blas(c), n, dT, n, 1, n, (const rocblas_int*)ip2, 1));
    PSX_HIP(hipGetLastError());
    trsm_left_dev(c, false, n, dB2, n, dT, n, n);   // dT = B2^{-1} dT
    trsm_left_dev(c, true, n, dB2, n, dT, n, n);
    transpose(c, n, dT, dY);
  } catch (...) {
    // nothing may still run on the caller's buffers once the error is out
    (void)hipStreamSynchronize(L2.s);
    (void)hipStreamSynchronize(c->stream);
    throw;
  }
  check_pivots(c, n, p1);
  if (!same) check_pivots(c, n, p2);
}

}  // namespace psx

using namespace psx;

extern "C" {

int psx_lu_solve(psx_ctx* hctx, int n, const double* A, int64_t lda, double* B,
                 int64_t ldb, int nrhs) {
  Ctx* c = reinterpret_cast<Ctx*>(hctx);
  return guarded(c, [&] {
    PSX_REQUIRE(n >= 1 && nrhs >= 0 && lda >= n && ldb >= n, PSX_ERR_ARGUMENT,
                "bad sizes for lu_solve");
    PSX_REQUIRE(A && (B || nrhs == 0), PSX_ERR_ARGUMENT, "null pointer");
    PSX_HIP(hipSetDevice(c->device));
    const size_t ab = sizeof(double) * n * (size_t)n,
                 bb = sizeof(double) * n * (size_t)std::max(nrhs, 1);
    XferBuf x(c, xfer_bytes({ab, bb}));
    double* dA = x.take(ab);
    double* dB = x.take(bb);
    h2d_matrix(c, dA, n, A, lda, n, n);
    if (nrhs > 0) h2d_matrix(c, dB, n, B, ldb, n, nrhs);
    lu_solve_dev(c, n, dA, n, dB, n, nrhs);
    if (nrhs > 0) d2h_matrix(c, B, ldb, dB, n, n, nrhs);
    PSX_HIP(hipStreamSynchronize(c->stream));
  });
}

int psx_lu_solve_pm(psx_ctx* hctx, int n, int sign, const double* Mpp, const double* Mmm,
                    int64_t ldM, double* B, int64_t ldb, int nrhs) {
  Ctx* c = reinterpret_cast<Ctx*>(hctx);
  return guarded(c, [&] {
    PSX_REQUIRE(n >= 1 && nrhs >= 1 && ldM >= n && ldb >= 2 * (int64_t)n, PSX_ERR_ARGUMENT,
                "bad sizes for lu_solve_pm");
    PSX_REQUIRE(sign == 1 || sign == -1, PSX_ERR_ARGUMENT, "sign must be +1 or -1");
    PSX_REQUIRE(Mpp && Mmm && B, PSX_ERR_ARGUMENT, "null pointer");
    PSX_REQUIRE(2 * (int64_t)n <= INT32_MAX / 2, PSX_ERR_ARGUMENT, "n too large");
    PSX_HIP(hipSetDevice(c->device));
    const int N = 2 * n;
    const size_t ab = sizeof(double) * N * (size_t)N, bb = sizeof(double) * N * (size_t)nrhs;
    XferBuf x(c, xfer_bytes({ab, bb}));
    double* dA = x.take(ab);
    double* dB = x.take(bb);
    // [M++ M--; M-- M++]: each block crosses the bus once, its twin is a
    // device copy
    const int64_t off = (int64_t)n * N + n;   // the bottom-right block
    h2d_matrix(c, dA, N, Mpp, ldM, n, n);
    h2d_matrix(c, dA + n, N, Mmm, ldM, n, n);
    PSX_HIP(hipMemcpy2DAsync(dA + off, sizeof(double) * N, dA, sizeof(double) * N,
                             sizeof(double) * n, n, hipMemcpyDeviceToDevice, c->stream));
    PSX_HIP(hipMemcpy2DAsync(dA + (int64_t)n * N, sizeof(double) * N, dA + n,
                             sizeof(double) * N, sizeof(double) * n, n,
                             hipMemcpyDeviceToDevice, c->stream));
    h2d_matrix(c, dB, N, B, ldb, N, nrhs);
    // [M++ -M--; -M-- M++] = D [M++ M--; M-- M++] D, D = diag(I, -I): solve
    // the first against D B and return D X
    const dim3 ng((unsigned)((n + 255) / 256), (unsigned)nrhs);
    if (sign < 0) {
      hipLaunchKernelGGL(negate_rows, ng, dim3(256), 0, c->stream, dB, (int64_t)N, n, n);
      PSX_HIP(hipGetLastError());
    }
    lu_solve_dev(c, N, dA, N, dB, N, nrhs);
    if (sign < 0) {
      hipLaunchKernelGGL(negate_rows, ng, dim3(256), 0, c->stream, dB, (int64_t)N, n, n);
      PSX_HIP(hipGetLastError());
    }
    d2h_matrix(c, B, ldb, dB, N, N, nrhs);
    PSX_HIP(hipStreamSynchronize(c->stream));
  });
}

int psx_lu_solve_d(psx_ctx* hctx, int n, double* dA, int64_t lda, double* dB, int64_t ldb,
                   int nrhs) {
  Ctx* c = reinterpret_cast<Ctx*>(hctx);
  return guarded(c, [&] {
    PSX_REQUIRE(n >= 1 && nrhs >= 0 && lda >= n && ldb >= n, PSX_ERR_ARGUMENT,
                "bad sizes for lu_solve");
    PSX_REQUIRE(dA && (dB || nrhs == 0), PSX_ERR_ARGUMENT, "null pointer");
    PSX_HIP(hipSetDevice(c->device));
    lu_solve_dev(c, n, dA, lda, dB, ldb, nrhs, true);
  });
}

int psx_lu_factor(psx_ctx* hctx, int n, const double* A, int64_t lda, double* LU, int64_t ldlu,
                  int* ipiv) {
  Ctx* c = reinterpret_cast<Ctx*>(hctx);
  return guarded(c, [&] {
    PSX_REQUIRE(n >= 1 && lda >= n && ldlu >= n, PSX_ERR_ARGUMENT, "bad sizes for lu_factor");
    PSX_REQUIRE(A && LU && ipiv, PSX_ERR_ARGUMENT, "null pointer");
    PSX_HIP(hipSetDevice(c->device));
    const size_t ab = sizeof(double) * n * (size_t)n, pb = sizeof(int) * ((size_t)n + 64);
    XferBuf x(c, xfer_bytes({ab, pb}));
    double* dA = x.take(ab);
    int* dp = reinterpret_cast<int*>(x.take(pb));
    h2d_matrix(c, dA, n, A, lda, n, n);
    lu_factor_dev(c, n, dA, n, dp, dp + n + 32);
    PSX_HIP(hipMemcpyAsync(ipiv, dp, sizeof(int) * n, hipMemcpyDeviceToHost, c->stream));
    d2h_matrix(c, LU, ldlu, dA, n, n, n);
    check_pivots(c, n, dp);
  });
}

int psx_decouple_covmat(psx_ctx* hctx, int n, const double* Y, const double* B1,
                        const double* B2, double* out) {
  Ctx* c = reinterpret_cast<Ctx*>(hctx);
  return guarded(c, [&] {
    PSX_REQUIRE(n >= 1, PSX_ERR_ARGUMENT, "n must be positive");
    PSX_REQUIRE(Y && B1 && B2 && out, PSX_ERR_ARGUMENT, "null pointer");
    PSX_HIP(hipSetDevice(c->device));
    // one matrix passed for both B1 and B2 is copied and factored once; B2 is
    // copied in while B1 is being factored
    const bool same = B1 == B2;
    const size_t nn = (size_t)n * n, b = sizeof(double) * nn;
    XferBuf x(c, xfer_bytes({4 * b}));
    double* d = x.take(4 * b);
    double* dB2 = same ? d + nn : d + 2 * nn;
    h2d_matrix(c, d + nn, n, B1, n, n, n);
    h2d_matrix(c, d, n, Y, n, n, n);
    decouple_dev(c, n, d, d + nn, dB2, d + 3 * nn,
                 [&] { h2d_matrix_x(c, dB2, n, B2, n, n, n); });
    d2h_matrix(c, out, n, d, n, n, n);
    PSX_HIP(hipStreamSynchronize(c->stream));
  });
}

}  // extern "C"
