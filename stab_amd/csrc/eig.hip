// Shift-invert Krylov-Schur eigensolver kernels (one work-group per point).
//
// Operator (temporal): T v = (A - sigma B)^-1 B v on the solver pencil, whose
// eigenvalues theta = 1/(omega - sigma) are largest for the omega nearest the
// shift.  Operator (spatial): the linearisation
//     [[C0,0],[0,I]] z = alpha [[-C1,-C2],[I,0]] z,  z = [phi; alpha phi]
// of the reference's companion (spatial.f90:982-1016); its shift-invert
// product reduces to one n x n solve with L(sigma) = C0 + sigma C1 + sigma^2 C2:
//     u = L(sigma)^-1 (-C1 z1 - C2 (z2 + sigma z1)),  T z = [u; z1 + sigma u].
// Solves use the LU factors (FP64, or equilibrated FP32 followed by FP64
// iterative-refinement steps whose residuals use the matrix-free pencil).
#include "bounds.h"
#include "pencil.h"

#define KS_MMAX 64
#define KS_NEVMAX 16

// Per-point Krylov-Schur state in global memory (small_off points here):
//   H  (KS_MMAX+1) x KS_MMAX, column-major, ld = KS_MMAX+1
//   Q  KS_MMAX x KS_MMAX (ld = KS_MMAX), Y KS_MMAX x KS_NEVMAX, theta[KS_MMAX]
#define SM_H 0
#define SM_Q ((KS_MMAX + 1) * KS_MMAX)
#define SM_Y (SM_Q + KS_MMAX * KS_MMAX)
#define SM_TH (SM_Y + KS_MMAX * KS_NEVMAX)
#define SM_SIZE (SM_TH + KS_MMAX)

struct KSState {
  int j0;        // first column to expand
  int k;         // kept columns after the last restart
  int done;      // 1: every wanted pair converged; 2: stopped on stagnation or NaN
  int cycles;
  double resmax; // max relative Ritz residual estimate of the wanted pairs
  double best;   // smallest resmax seen
  int stall;     // cycles without a 10x improvement of best
  int irbad;     // 1 if a refined solve contracted poorly (FP32 factors inadequate)
  int steps;     // operator applications so far
  int pad;
};

// ---------------------------------------------------------------------------
// y <- M^-1 y with the factors of k_lu and the 64 x 64 diagonal-block
// inverses of k_blkinv (scales applied by the caller).  The solve reads the
// whole factor once and is bound by how many bytes one work-group keeps in
// flight, so every load is 16 bytes wide (two FP32 or one FP64 complex matrix
// entries of consecutive rows) and each lane issues 16 of them before using
// any (64 KB in flight per work-group).  The factor and block inverses are
// read with streaming (non-temporal) loads: a point's next solve comes after
// the other work-groups have streamed theirs, so they would only push the
// operators D1, D2, which every pencil product rereads, out of L2.  Per block
// of 64 rows:
//   1. y_top <- inv(D) y_top: lane (i, q) sums columns 16q..16q+15 of row i
//      of the column-major inverse (a wave reads 64 consecutive entries per
//      load); the four partial sums meet in tmp (NT = 256 entries);
//   2. the rows below (forward) or above (backward): a row group g is E rows
//      (E = 16 bytes / entry size); the 16 lanes of a DPP row take 16
//      consecutive groups, the four DPP rows of a wave the four quarters q of
//      the 64 columns, and the quarters are summed across the rows.  Consecutive
//      lanes so read consecutive 16-byte entries; with the quarters on
//      consecutive lanes instead every group of four lanes met four cache
//      lines, and a CU could not take in more than 13 bytes a cycle, at any
//      number of loads in flight.
// Columns of a partial last block (bs < 64) beyond bs are never loaded.
// y, work in LDS (npad); tmp in LDS (NT entries).
// ---------------------------------------------------------------------------
#define SOLVE_BS 64
template <typename T> struct Row16;
template <> struct Row16<float> {
  typedef float V __attribute__((ext_vector_type(4)));
  static constexpr int E = 2;
  __device__ static zd get(const V &v, int e) { return e == 0 ? mk((double)v.x, (double)v.y) : mk((double)v.z, (double)v.w); }
};
template <> struct Row16<double> {
  typedef double V __attribute__((ext_vector_type(2)));
  static constexpr int E = 1;
  __device__ static zd get(const V &v, int) { return mk(v.x, v.y); }
};

// For each right-hand side r < NR: tmp[r NT + 0..bs) <- inv(D) y_r[k0..k0+bs)
// with D the diagonal block at inv (column major, entries beyond bs zero),
// tmp[r NT + bs..64) <- 0, and y_r[k0..k0+bs) <- the same.  The inverse is
// loaded once for all right-hand sides.  Branch-free: indexes past bs are
// clamped to bs - 1 and meet zero entries.  Two barriers.
template <typename T, int NT, int NR>
__device__ inline void solve_diag(const cx<T> *__restrict__ inv, int k0, int bs, zd *const (&y)[NR], zd *tmp) {
  constexpr int BS = SOLVE_BS;
  const int t = threadIdx.x, i = t & (BS - 1), q = t >> 6;
  const cx<T> *col = inv + (size_t)(q * 16) * BS + i;
  cx<T> v[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) v[j] = load_stream(col + j * BS);
  zd s[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) s[r] = czero<double>();
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const zd vj = cvt<double>(v[j]);
    const int kk = k0 + min(q * 16 + j, bs - 1);
#pragma unroll
    for (int r = 0; r < NR; ++r) s[r] = cfma(s[r], vj, y[r][kk]);
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) tmp[r * NT + t] = s[r];
  __syncthreads();
  if (t < BS) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      zd *tr = tmp + r * NT;
      const zd v = tr[t] + tr[BS + t] + tr[2 * BS + t] + tr[3 * BS + t];
      tr[t] = (t < bs) ? v : czero<double>();
      if (t < bs) y[r][k0 + t] = v;
    }
  }
  __syncthreads();
}

// y_r[r0..r1) -= A[r0..r1, k0..k0+bs) tmp[r NT + 0..bs) for r < NR (the matrix
// is loaded once for all right-hand sides); r0, r1 multiples of E.  PIPE
// (the inverse-iteration kernels) issues each entry's load for the next pass
// as soon as the entry is used, so loads stay in flight through the arithmetic
// and the reductions; the other kernels, tighter on registers, load pass by
// pass.  The arithmetic is the same either way.
// Branch-free: rows past r1 take the last row group (not written back).
template <typename T, int NT, int NR, bool PIPE = false>
__device__ inline void solve_update(const cx<T> *__restrict__ A, int lda, int k0, int bs, int r0, int r1,
                                    zd *const (&y)[NR], const zd *tmp) {
  typedef Row16<T> R;
  typedef typename R::V V;
  constexpr int E = R::E, G = NT / 4;        // G row groups of E rows per pass
  const int t = threadIdx.x, q = (t >> 4) & 3, g = (t >> 6) * 16 + (t & 15);
  const int ldv = lda / E;
  // bs is 32 or 64: the upper columns of a 32-wide last block meet zeros of
  // tmp, from columns in range.  32-bit lane offsets from uniform bases.
  const int col = k0 + (q * 16 < bs ? q * 16 : q * 16 - 32);
  auto offset = [&](int rb) { return (unsigned)((col * ldv + min(rb + g * E, r1 - E) / E) * (int)sizeof(V)); };
  auto entry = [&](int j, unsigned off) {
    return __builtin_nontemporal_load((const V *)((const char *)A + (size_t)j * ldv * sizeof(V) + off));
  };
  V v[16];
  auto load = [&](int rb) {
    const unsigned off = offset(rb);
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = entry(j, off);
  };
  // one pass over rows rb .. rb + G E; with NEXT, each entry's register is
  // reloaded with the next pass's entry (rows rn ..) as soon as it is used
  auto pass = [&](int rb, int rn, auto next) {
    constexpr bool NEXT = decltype(next)::value;
    const int row = rb + g * E;
    const unsigned off = offset(rn);
    zd a[NR][E];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int e = 0; e < E; ++e) a[r][e] = czero<double>();
#pragma unroll
    for (int j = 0; j < 16; ++j) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const zd mj = tmp[r * NT + q * 16 + j];
#pragma unroll
        for (int e = 0; e < E; ++e) a[r][e] = cfma(a[r][e], R::get(v[j], e), mj);
      }
      if (NEXT) v[j] = entry(j, off);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int e = 0; e < E; ++e) {
        a[r][e].x = add_rows<32>(add_rows<16>(a[r][e].x));
        a[r][e].y = add_rows<32>(add_rows<16>(a[r][e].y));
      }
    if (row < r1 && q == 0) {
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int e = 0; e < E; ++e) y[r][row + e] = y[r][row + e] - a[r][e];
    }
  };
  if (!PIPE) {
#pragma unroll 1
    for (int rb = r0; rb < r1; rb += G * E) {
      load(rb);
      pass(rb, rb, std::false_type());
    }
    return;
  }
  // the next pass's loads go out while this pass computes (in the registers
  // this pass has just used, so no second buffer)
  if (r0 >= r1) return;
  load(r0);
  int rb = r0;
#pragma unroll 1
  for (; rb + G * E < r1; rb += G * E) pass(rb, rb + G * E, std::true_type());
  pass(rb, rb, std::false_type());
}

// NR right-hand sides y[r] (LDS, npad) solved together; tmp holds NR NT
// entries, work npad.
template <typename T, int NT, int NR, bool PIPE = false>
__device__ __forceinline__ void lu_solve_n(const PointDev &P, const cx<T> *__restrict__ A, const int *__restrict__ ipiv,
                                           const cx<T> *__restrict__ blk, zd *const (&y)[NR], zd *tmp, zd *work) {
  static_assert(NT == 4 * SOLVE_BS, "four lanes per row of a 64-row block");
  static_assert(LU_PREC == 1 + 4 * SOLVE_BS, "one interchange record per 64-row block");
  constexpr int BS = SOLVE_BS;
  const int n = P.npad, lda = P.npad, t = threadIdx.x;
  const int *perm = ipiv + n;
  const int nblk = (n + BS - 1) / BS;
  const cx<T> *Li = blk, *Ui = blk + (size_t)nblk * BS * BS;   // layout of k_blkinv
  const int *rec0 = ipiv + 2 * n;                                // pivot mode, block records
  const bool progressive = rec0[0] != 0;
  if (!progressive) {
    // y <- P y (one gather through `work` per right-hand side)
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      for (int i = t; i < n; i += NT) work[i] = y[r][perm[i]];
      __syncthreads();
      for (int i = t; i < n; i += NT) y[r][i] = work[i];
      __syncthreads();
    }
  }
  for (int b = 0; b < nblk; ++b) {
    const int k0 = b * BS, bs = min(BS, n - k0);
    if (progressive) {
      // the block's net interchanges (rows >= k0, at most 2 BS of them and
      // never more than n - k0, so they fit in work)
      const int *rec = rec0 + 1 + (size_t)b * LU_PREC;
      const int ns = rec[0];
      if (ns > 0) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          for (int e = t; e < ns; e += NT) work[e] = y[r][rec[1 + 2 * BS + e]];
          __syncthreads();
          for (int e = t; e < ns; e += NT) y[r][rec[1 + e]] = work[e];
          __syncthreads();
        }
      }
    }
    solve_diag<T, NT, NR>(Li + (size_t)b * BS * BS, k0, bs, y, tmp);
    if (k0 + bs < n) {
      solve_update<T, NT, NR, PIPE>(A, lda, k0, bs, k0 + bs, n, y, tmp);
      __syncthreads();
    }
  }
  for (int b = nblk - 1; b >= 0; --b) {
    const int k0 = b * BS, bs = min(BS, n - k0);
    solve_diag<T, NT, NR>(Ui + (size_t)b * BS * BS, k0, bs, y, tmp);
    if (k0 > 0) {
      solve_update<T, NT, NR, PIPE>(A, lda, k0, bs, 0, k0, y, tmp);
      __syncthreads();
    }
  }
}

// The value of lane l (the same l in every lane).
__device__ inline double lane_get(double x, int l) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)(unsigned int)(b & 0xffffffffLL), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned int)hi << 32) | (unsigned int)lo));
}
__device__ inline zd lane_get(zd x, int l) { return mk(lane_get(x.x, l), lane_get(x.y, l)); }
// Sum over the wave, in every lane (row shifts, then row broadcasts; lanes
// without a source add nothing).
template <int CTRL, int RM> __device__ inline double dpp_or_zero(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned int)(b & 0xffffffffLL), CTRL, RM, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, RM, 0xF, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned int)hi << 32) | (unsigned int)lo));
}
__device__ inline double wave_sum(double x) {
  x += dpp_or_zero<0x111, 0xF>(x);
  x += dpp_or_zero<0x112, 0xF>(x);
  x += dpp_or_zero<0x114, 0xF>(x);
  x += dpp_or_zero<0x118, 0xF>(x);
  x += dpp_or_zero<0x142, 0xA>(x);
  x += dpp_or_zero<0x143, 0xC>(x);
  return lane63(x);
}

// The same solve for work-groups of more than four waves, for batches that
// leave CUs idle (at most a work-group per CU): what bounds it then is the
// chain of 2 nblk block steps, not memory, so
//   * NT / 4 row groups x 64 columns are in flight at once, and every register
//     of a pass is reloaded, as soon as it is used, with the entry of the next
//     pass, across block steps too: the loads of a step do not depend on the
//     solution, so they are on their way while the step before is finished.
//     The compiled loop waits for all of them, and for those of the inverse,
//     issued last, at the head of each pass, so part of a memory latency is
//     still met in every pass;
//   * the same holds for the entries of the diagonal-block inverse (four waves,
//     its quarters on the DPP rows, no partial sums in LDS) and for the
//     interchange record (one entry per thread);
//   * a step has two barriers (four with interchanges).
// Every sum is formed in the order of lu_solve_n, so the result is the same.
// One point of N = 96 in FP64 (n = 480, 3.7 MB): 134 us with 256 threads,
// 52 us with 512.  The factor comes with plain loads: at these batch sizes
// it can stay in the caches from one solve to the next.  kb is 32 or 64: the
// lanes of the upper columns of a 32-wide last block take in-range columns
// and meet the zeros of tmp.
template <typename T, int NT, int NR>
__device__ __forceinline__ void lu_solve_wide(const PointDev &P, const cx<T> *__restrict__ A, const int *__restrict__ ipiv,
                                              const cx<T> *__restrict__ blk, zd *const (&y)[NR], zd *tmp) {
  typedef Row16<T> R;
  typedef typename R::V V;
  constexpr int BS = SOLVE_BS, E = R::E, G = NT / 4, CPL = 16;
  static_assert(NT >= 4 * BS, "four waves for the diagonal product");
  const int n = P.npad, lda = P.npad, t = threadIdx.x;
  const int nblk = (n + BS - 1) / BS, q = (t >> 4) & 3, g = (t >> 6) * 16 + (t & 15), ldv = lda / E;
  const bool dwave = __builtin_amdgcn_readfirstlane(t >> 6) < 4;     // waves of the diagonal product
  const int dr = g & (BS - 1);                                        // its row; q its quarter of the columns
  const int *rec0 = ipiv + 2 * n;
  const bool progressive = rec0[0] != 0;
  if (!progressive) {
    const int *perm = ipiv + n;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      zd w[(1280 + NT - 1) / NT];
#pragma unroll
      for (int k = 0; k < (1280 + NT - 1) / NT; ++k) if (t + k * NT < n) w[k] = y[r][perm[t + k * NT]];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < (1280 + NT - 1) / NT; ++k) if (t + k * NT < n) y[r][t + k * NT] = w[k];
      __syncthreads();
    }
  }
  // first row of pass 0 and end row of step s (forward steps 0 .. nblk - 1,
  // then backward over the blocks nblk - 1 .. 0)
  auto rows = [&](int s, int &k0, int &r0, int &r1) {
    const int b = s < nblk ? s : 2 * nblk - 1 - s;
    k0 = b * BS;
    r0 = s < nblk ? min(k0 + BS, n) : 0;
    r1 = s < nblk ? n : k0;
  };
  // Byte offsets of this lane's first entry of a pass and of its first column
  // of the step's diagonal inverse: 32-bit lane offsets from bases that are the
  // same for the work-group, so sixteen loads need no lane addresses of their own.
  auto entry = [&](int k0, int rb, int r1) {
    const int qc = (k0 + q * 16 < n) ? q * 16 : q * 16 - 32;
    return (unsigned)(((k0 + qc) * ldv + max(min(rb + g * E, r1 - E), 0) / E) * (int)sizeof(V));
  };
  auto load_v = [&](int j, unsigned off) { return *(const V *)((const char *)A + (size_t)j * ldv * sizeof(V) + off); };
  const unsigned doff = (unsigned)((q * CPL * BS + dr) * (int)sizeof(cx<T>));
  auto inv_base = [&](int s) {
    const int b = s < nblk ? s : 2 * nblk - 1 - s;
    return (const char *)(blk + ((size_t)(s < nblk ? 0 : nblk) + b) * BS * BS);
  };
  auto load_d = [&](int j, const char *c) { return *(const cx<T> *)(c + (size_t)j * BS * sizeof(cx<T>) + doff); };
  auto records = [&](int s, int &ns, int &src, int &dst) {
    const int *rec = rec0 + 1 + (size_t)min(s, nblk - 1) * LU_PREC;
    ns = rec[0];
    const int e = min(t, 2 * BS - 1);
    dst = rec[1 + e];
    src = rec[1 + 2 * BS + e];
  };
  int k0, r0, r1, ns = 0, src = 0, dst = 0;
  rows(0, k0, r0, r1);
  V v[16];
  cx<T> d[CPL];
  {
    const unsigned p = entry(k0, r0, r1);
    const char *c = inv_base(0);
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = load_v(j, p);
    if (dwave) {
#pragma unroll
      for (int j = 0; j < CPL; ++j) d[j] = load_d(j, c);
    }
  }
  if (progressive) records(0, ns, src, dst);
#pragma unroll 1
  for (int s = 0; s < 2 * nblk; ++s) {
    const int bs = min(BS, n - k0);
    if (progressive && s < nblk) {
      if (ns > 0) {                                     // at most 2 BS <= NT entries
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          zd w = czero<double>();
          if (t < ns) w = y[r][src];
          __syncthreads();
          if (t < ns) y[r][dst] = w;
        }
        __syncthreads();
      }
      records(s + 1, ns, src, dst);
    }
    int k0n = k0, r0n = r0, r1n = r1;
    if (s + 1 < 2 * nblk) rows(s + 1, k0n, r0n, r1n);
    if (dwave) {
      const char *c = inv_base(min(s + 1, 2 * nblk - 1));
      zd a[NR];
#pragma unroll
      for (int r = 0; r < NR; ++r) a[r] = czero<double>();
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        const int kk = k0 + min(q * CPL + j, bs - 1);  // entries past bs are zero
#pragma unroll
        for (int r = 0; r < NR; ++r) a[r] = cfma(a[r], cvt<double>(d[j]), y[r][kk]);
        d[j] = load_d(j, c);
      }
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        a[r] = mk(sum_rows_in_order(a[r].x), sum_rows_in_order(a[r].y));
        // tmp, not y: other rows of the block still read y
        if (q == 0) tmp[r * BS + dr] = (dr < bs) ? a[r] : czero<double>();
      }
    }
    __syncthreads();
    if (t < NR * BS && (t & (BS - 1)) < bs) (t < BS ? y[0] : y[NR - 1])[k0 + (t & (BS - 1))] = tmp[t];
    static_assert(NR <= 2, "one or two right-hand sides");
#pragma unroll 1
    for (int rb = r0; rb < r1; rb += G * E) {
      const bool last = rb + G * E >= r1;
      const unsigned p = last ? entry(k0n, r0n, r1n) : entry(k0, rb + G * E, r1);
      zd a[NR][E];
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int e = 0; e < E; ++e) a[r][e] = czero<double>();
#pragma unroll
      for (int j = 0; j < 16; ++j) {
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const zd mj = tmp[r * BS + q * 16 + j];
#pragma unroll
          for (int e = 0; e < E; ++e) a[r][e] = cfma(a[r][e], R::get(v[j], e), mj);
        }
        v[j] = load_v(j, p);
      }
      const int row = rb + g * E;
#pragma unroll
      for (int r = 0; r < NR; ++r)
#pragma unroll
        for (int e = 0; e < E; ++e) {
          a[r][e].x = add_rows<32>(add_rows<16>(a[r][e].x));
          a[r][e].y = add_rows<32>(add_rows<16>(a[r][e].y));
        }
      if (row < r1 && q == 0) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int e = 0; e < E; ++e) y[r][row + e] = y[r][row + e] - a[r][e];
      }
    }
    if (r0 >= r1) {                                     // nothing to update: fetch the next step's first pass
      const unsigned p = entry(k0n, r0n, r1n);
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = load_v(j, p);
    }
    __syncthreads();
    k0 = k0n; r0 = r0n; r1 = r1n;
  }
}

template <typename T, int NT, int NR, bool PIPE = false>
__device__ __forceinline__ void lu_solve_many(const PointDev &P, const cx<T> *__restrict__ A, const int *__restrict__ ipiv,
                                              const cx<T> *__restrict__ blk, zd *const (&y)[NR], zd *tmp, zd *work) {
  if constexpr (NT > 256) lu_solve_wide<T, NT, NR>(P, A, ipiv, blk, y, tmp);
  else lu_solve_n<T, NT, NR, PIPE>(P, A, ipiv, blk, y, tmp, work);
}

template <typename T, int NT, bool PIPE = false>
__device__ __forceinline__ void lu_solve(const PointDev &P, const cx<T> *__restrict__ A, const int *__restrict__ ipiv,
                                         const cx<T> *__restrict__ blk, zd *y, zd *tmp, zd *work) {
  zd *const ys[1] = {y};
  lu_solve_many<T, NT, 1, PIPE>(P, A, ipiv, blk, ys, tmp, work);
}

// Block-wide reduction of NV complex partial sums; result broadcast to all.
// Partial sums come from the first RT = 256 threads (red_first, RT), so
// the result does not depend on the size of the work-group.
__device__ inline int red_first() { return threadIdx.x < 256 ? (int)threadIdx.x : 1 << 30; }
constexpr int RT = 256;
template <int NT, int NV>
__device__ void block_reduce(zd (&v)[NV], zd *red) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  if (NT <= RT || w < RT / 64) {
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = mk(wave_sum_xor(v[k].x), wave_sum_xor(v[k].y));
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < NV; ++k) red[w * NV + k] = v[k];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    zd s = czero<double>();
#pragma unroll
    for (int ww = 0; ww < RT / 64; ++ww) s = s + red[ww * NV + k];
    v[k] = s;
  }
  __syncthreads();
}

template <int NT>
__device__ double block_norm2(const zd *x, int len, zd *red) {
  zd v[1] = {czero<double>()};
  for (int r = red_first(); r < len; r += RT) v[0].x += abs2(x[r]);
  block_reduce<NT, 1>(v, red);
  return v[0].x;
}

// First index of largest value over the work-group: (v, i) per thread, v = -1
// where it has none (a NaN never becomes a candidate); red: NT / 64 entries.
template <int NT>
__device__ int block_argmax(double v, int i, zd *red) {
  const int t = threadIdx.x;
  wave_argmax(v, i);
  if ((t & 63) == 0) red[t >> 6] = mk(v, (double)i);
  __syncthreads();
#pragma unroll 4
  for (int w = 0; w < NT / 64; ++w) {
    const zd c = red[w];
    if (c.x > v || (c.x == v && (int)c.y < i)) { v = c.x; i = (int)c.y; }
  }
  __syncthreads();
  return i;
}

// Shared-memory layout of the operator kernels (dynamic LDS, zd units).
// The full layout serves refinement and the spatial operator; the compact one
// (plain FP64, temporal only) keeps just the solve vector and the Krylov
// vector, so more work-groups fit on a CU.
struct OpLds {
  zd *y, *rhs, *res, *X1, *X2, *z, *red, *tmp, *w2;
  // nvecmax: longest Krylov vector (2 n for spatial points).  w2, the gather
  // buffer of the solves, aliases X1/X2 (10 ny >= npad), which are idle then.
  // red: NT / 64 sums of up to 8 values; tmp: NT entries (256 threads) or 64
  // per right-hand side.
  __device__ OpLds(zd *base, int nt, int npadmax, int nymax, int full, int nvecmax) {
    red = base;
    tmp = red + (nt > 256 ? 128 : 64);
    y = base + 320;
    z = y + npadmax;
    if (full) {
      rhs = z + nvecmax;
      res = rhs + npadmax;
      X1 = res + npadmax;
      X2 = X1 + 5 * nymax;
      w2 = X1;
    } else {
      rhs = res = X1 = X2 = w2 = nullptr;
    }
  }
};

__host__ __device__ inline size_t op_lds_bytes(int npadmax, int nymax, int full, int nvecmax) {
  return sizeof(zd) * (320 + (size_t)npadmax + (size_t)nvecmax +
                       (full ? 2 * (size_t)npadmax + 10 * (size_t)nymax : 0));
}

// y = M^-1 rhs in FP64 quality: scaled solve with the factors, then
// iterative-refinement steps with the FP64 matrix-free shifted pencil.
// ir > 0: exactly ir steps.  ir < 0: adaptive, at most -ir steps, stopping once
// the correction is below 1e-14 of the solution or stops shrinking by half
// (the FP64 rounding floor of the residual has been reached).  The contraction
// per step is about kappa(M) u32.
template <typename T, int NB, int NT, bool PIPE = false>
__device__ bool shifted_solve(const PointDev &P, const cx<T> *A, const int *ipiv, const cx<T> *Lb, const cx<T> *Ub,
                              const double *dr, const double *dc, const zd *coef, const double *ops, int ir,
                              OpLds &L) {
  const int n = P.npad, t = threadIdx.x;
  for (int r = t; r < n; r += NT) L.y[r] = (r < P.n) ? L.rhs[r] * dr[r] : czero<double>();
  __syncthreads();
  lu_solve<T, NT, PIPE>(P, A, ipiv, Lb, L.y, L.tmp, L.w2);
  for (int r = t; r < n; r += NT) L.y[r] = L.y[r] * dc[r];
  __syncthreads();
  const bool adaptive = ir < 0;
  const int steps = adaptive ? -ir : ir;
  double dprev = 0.0;
  bool ok = !adaptive;
  for (int s = 0; s < steps; ++s) {
    pencil_apply<NT>(P, coef, ops, FORM_SHIFTED, P.shift, L.y, L.res, L.X1, L.X2, L.red);
    for (int r = t; r < n; r += NT) L.res[r] = (r < P.n) ? (L.rhs[r] - L.res[r]) * dr[r] : czero<double>();
    __syncthreads();
    lu_solve<T, NT, PIPE>(P, A, ipiv, Lb, L.res, L.tmp, L.w2);
    zd nrm[2] = {czero<double>(), czero<double>()};
    for (int r = red_first(); r < n; r += RT) {
      const zd d = L.res[r] * dc[r];
      L.y[r] = L.y[r] + d;
      nrm[0].x += abs2(d);
      nrm[1].x += abs2(L.y[r]);
    }
    if (adaptive) {
      block_reduce<NT, 2>(nrm, L.red);
      // the FP32 factors are adequate for this shift when the first correction
      // is below 1e-2 of the solution (refinement then contracts fast)
      if (s == 0) ok = nrm[0].x <= 1e-4 * nrm[1].x;
      if (nrm[0].x <= 1e-28 * nrm[1].x || (s > 0 && nrm[0].x > 0.25 * dprev)) break;
      dprev = nrm[0].x;
    } else {
      __syncthreads();
    }
  }
  return ok;
}

// w = T v for point P; v read from global (length nvec), w left in L.z.
// FULL = false compiles only the plain FP64 temporal operator.
template <typename T, int NB, int NT, bool FULL = true>
__device__ bool apply_op(const PointDev &P, const cx<T> *A, const int *ipiv, const cx<T> *Lb, const cx<T> *Ub,
                         const double *dr, const double *dc, const zd *coef, const double *ops, int ir,
                         const zd *v, OpLds &L) {
  const int n = P.n, t = threadIdx.x;
  if (!FULL || (P.itype == 1 && L.rhs == nullptr)) {
    // plain FP64 temporal: y = B v in place, one solve, no scaling
    for (int r = t; r < n; r += NT) L.z[r] = v[r];
    __syncthreads();
    pencil_apply<NT>(P, coef, ops, FORM_BM, P.shift, L.z, L.y, L.X1, L.X2, L.red);
    for (int r = n + t; r < P.npad; r += NT) L.y[r] = czero<double>();
    __syncthreads();
    lu_solve<T, NT>(P, A, ipiv, Lb, L.y, L.tmp, L.z);
    for (int r = t; r < n; r += NT) L.z[r] = L.y[r];
    __syncthreads();
    return true;
  }
  if constexpr (!FULL) return true;
  bool ok;
  if (P.itype == 1) {
    for (int r = t; r < n; r += NT) L.z[r] = v[r];
    __syncthreads();
    pencil_apply<NT>(P, coef, ops, FORM_BM, P.shift, L.z, L.rhs, L.X1, L.X2, L.red);
    ok = shifted_solve<T, NB, NT>(P, A, ipiv, Lb, Ub, dr, dc, coef, ops, ir, L);
    for (int r = t; r < n; r += NT) L.z[r] = L.y[r];
    __syncthreads();
  } else {
    const zd sg = P.shift;
    // z holds [z1; z2 + sigma z1]
    for (int r = t; r < n; r += NT) { L.z[r] = v[r]; L.z[n + r] = v[n + r] + sg * v[r]; }
    __syncthreads();
    pencil_apply<NT>(P, coef, ops, FORM_C1, sg, L.z, L.rhs, L.X1, L.X2, L.red);
    pencil_apply<NT>(P, coef, ops, FORM_C2, sg, L.z + n, L.res, L.X1, L.X2, L.red);
    for (int r = t; r < n; r += NT) L.rhs[r] = czero<double>() - L.rhs[r] - L.res[r];
    __syncthreads();
    ok = shifted_solve<T, NB, NT>(P, A, ipiv, Lb, Ub, dr, dc, coef, ops, ir, L);
    for (int r = t; r < n; r += NT) { L.z[n + r] = L.z[r] + sg * L.y[r]; L.z[r] = L.y[r]; }
    __syncthreads();
  }
  return ok;
}

// Deterministic start vector: T applied to a hashed pseudo-random vector.
__device__ inline double hash01(unsigned a, unsigned b) {
  unsigned h = a * 0x9E3779B1u ^ (b + 0x7F4A7C15u) * 0x85EBCA77u;
  h ^= h >> 15; h *= 0x2C1B3C6Du; h ^= h >> 12; h *= 0x297A2D39u; h ^= h >> 15;
  return (double)h * (1.0 / 4294967296.0) - 0.5;
}

// Seed of a point's start vector from the point's own parameters, so that its
// iterates do not depend on where it sits in the batch.
__device__ inline unsigned point_seed(const PointDev &P) {
  const double f[] = {P.alpha.x, P.alpha.y, P.beta.x, P.beta.y, P.omega.x, P.omega.y, P.shift.x, P.shift.y,
                      P.Re, P.Ma, P.Pr, P.Te, P.yi, P.ymax};
  unsigned long long h = 0xCBF29CE484222325ull ^ (unsigned long long)(P.ny * 4 + P.itype);
#pragma unroll
  for (int k = 0; k < (int)(sizeof(f) / sizeof(f[0])); ++k) {
    h ^= (unsigned long long)__double_as_longlong(f[k]);
    h *= 0x100000001B3ull;
    h ^= h >> 29;
  }
  return (unsigned)(h ^ (h >> 32));
}

// ---------------------------------------------------------------------------
// Arnoldi expansion from column j0 to m (CGS2).  V column-major, ld = ldv.
// ---------------------------------------------------------------------------
template <typename T, int NB, int NT, bool FULL, bool GS4 = false>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(FULL || NT > 256 ? 2 : 3))) void k_arnoldi(const PointDev *__restrict__ pts, const cx<T> *__restrict__ mats,
                                                const int *__restrict__ pivs, const cx<T> *__restrict__ blks,
                                                const double *__restrict__ scales, const zd *__restrict__ coef,
                                                const double *__restrict__ ops, zd *__restrict__ Vall,
                                                zd *__restrict__ small, KSState *__restrict__ st, int m, int ir,
                                                int npadmax, int nymax, int nvecmax, int start) {
  extern __shared__ zd lds[];
  const PointDev &P = pts[blockIdx.x];
  if (st[blockIdx.x].done) return;
  int j0 = st[blockIdx.x].j0;
  OpLds L(lds, NT, npadmax, nymax, FULL ? 1 : 0, nvecmax);
  const int t = threadIdx.x, nv = P.nvec;
  const size_t ldv = (size_t)nv;
  zd *V = Vall + P.vec_off;
  zd *H = small + P.small_off + SM_H;
  const int ldh = KS_MMAX + 1;
  const cx<T> *A = mats + P.mat_off;
  const int *ipiv = pivs + P.piv_off;
  const cx<T> *Lb = blks + P.blk_off, *Ub = nullptr;
  const double *dr = scales + P.scale_off, *dc = dr + P.npad;

  bool allok = true;
  if (start) {
    // v0 = T r / ||T r||, r pseudo-random
    const unsigned seed = point_seed(P);
    for (int r = t; r < nv; r += NT) V[r] = mk(hash01(seed, 2 * r), hash01(seed, 2 * r + 1));
    __threadfence_block();
    __syncthreads();
    allok &= apply_op<T, NB, NT, FULL>(P, A, ipiv, Lb, Ub, dr, dc, coef, ops, ir, V, L);
    const double nrm = sqrt(block_norm2<NT>(L.z, nv, L.red));
    for (int r = t; r < nv; r += NT) V[r] = L.z[r] * (1.0 / nrm);
    for (int e = t; e < ldh * KS_MMAX; e += NT) H[e] = czero<double>();
    __syncthreads();
    j0 = 0;
  }
  for (int j = j0; j < m; ++j) {
    allok &= apply_op<T, NB, NT, FULL>(P, A, ipiv, Lb, Ub, dr, dc, coef, ops, ir, V + (size_t)j * ldv, L);
    // two passes of classical Gram-Schmidt against V[:, 0..j], all
    // coefficients of a pass at once: a wave per column forms h_l, then a
    // thread per row subtracts the whole combination (two barriers a pass;
    // groups of four columns with a block reduction each took 37 us a step at
    // n = 480, 14 us here)
    if constexpr (GS4) {
      for (int pass = 0; pass < 2; ++pass) {
        for (int l0 = 0; l0 <= j; l0 += 4) {
          zd h[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) h[k] = czero<double>();
          for (int r = red_first(); r < nv; r += RT) {
            const zd w = L.z[r];
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (l0 + k <= j) h[k] = cfmac(h[k], V[(size_t)(l0 + k) * ldv + r], w);
          }
          block_reduce<NT, 4>(h, L.red);
          for (int r = t; r < nv; r += NT) {
            zd w = L.z[r];
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (l0 + k <= j) w = cfms(w, V[(size_t)(l0 + k) * ldv + r], h[k]);
            L.z[r] = w;
          }
          if (t < 4 && l0 + t <= j) {
            zd hv = h[0];
#pragma unroll
            for (int k = 0; k < 4; ++k) if (k == t) hv = h[k];
            H[(size_t)j * ldh + l0 + t] = H[(size_t)j * ldh + l0 + t] + hv;
          }
          __syncthreads();
        }
      }
    } else
    for (int pass = 0; pass < 2; ++pass) {
      for (int l = t >> 6; l <= j; l += NT / 64) {
        const zd *Vl = V + (size_t)l * ldv + (t & 63), *z = L.z + (t & 63);
        zd s = czero<double>();
        for_loaded<8>((nv - (t & 63) + 63) / 64, [&](int r) { return Vl[64 * r]; },
                      [&](int r, zd v) { s = cfmac(s, v, z[64 * r]); });
        s = mk(wave_sum(s.x), wave_sum(s.y));
        if ((t & 63) == 0) {
          L.tmp[l] = s;
          H[(size_t)j * ldh + l] = H[(size_t)j * ldh + l] + s;
        }
      }
      __syncthreads();
      for (int r = t; r < nv; r += NT) {
        zd w = L.z[r];
        for_loaded<8>(j + 1, [&](int l) { return V[(size_t)l * ldv + r]; },
                      [&](int l, zd v) { w = cfms(w, v, L.tmp[l]); });
        L.z[r] = w;
      }
      __syncthreads();
    }
    double nrm = sqrt(block_norm2<NT>(L.z, nv, L.red));
    if (!(nrm > 1e-300)) nrm = 1e-300;
    for (int r = t; r < nv; r += NT) V[(size_t)(j + 1) * ldv + r] = L.z[r] * (1.0 / nrm);
    if (t == 0) H[(size_t)j * ldh + j + 1] = mk(nrm, 0.0);
    __syncthreads();
  }
  if (t == 0) {
    st[blockIdx.x].steps += (m - j0) + (start ? 1 : 0);
    st[blockIdx.x].j0 = m;
    if (start) st[blockIdx.x].k = 0;
    if (!allok) st[blockIdx.x].irbad = 1;
  }
}

// ---------------------------------------------------------------------------
// Small dense eigenproblem of H_m: Householder reduction to Hessenberg form,
// complex single-shift QR to Schur form T = Q^H H Q, then the `keep`
// eigenvalues of largest modulus are moved to the leading positions in
// decreasing modulus.  Ritz vectors of the first nev, residual estimates and
// convergence are written back.
//
// One work-group of two waves per point: wave 0 works on H, wave 1 applies the
// rotations of each finished sweep to Q while wave 0 runs the next (two
// rotation lists, one barrier a sweep).  The step is a chain of some 2500
// dependent rotations (m = 40), so what counts is the latency of one.  A sweep
// therefore runs in two phases.  Lane j owns column j while the rotations are
// found: it carries its entry of the current row in a register and reads the
// next row ahead, and the 3 x 3 window that determines the next rotation is
// held by every lane, so no rotation waits for LDS.  Then lane i owns row i
// and applies the sweep's rotations to the columns in one pass.  With a lone
// wave, LDS round trips and library hypot calls in every rotation a point
// took 2.95 ms (m = 40) and 1.09 ms (m = 24); this form takes 1.21 and 0.52 ms,
// some 780 cycles a rotation in phase 1 (about 55 FP64 operations, mostly
// dependent) and 220 in phase 2.
// ---------------------------------------------------------------------------
// Order LDS accesses of one wave's lanes (a wave's LDS operations execute in
// order; this keeps the compiler to it).
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Rotation with c x + s y = r, c y - conj(s) x = 0, c real, the same (x, y) in
// every lane.  Squares that would under- or overflow, and x = 0, take the
// scaled form.
__device__ inline void givens(zd x, zd y, double &c, zd &s) {
  const double x2 = abs2(x), n2 = x2 + abs2(y);
  const double rx = rsqrt(x2), f = rx * rsqrt(n2);
  c = x2 * f;
  s = x * conj(y) * f;
  if (__builtin_expect(!(x2 > 1e-280 && n2 < 1e280), 0)) {
    const double big = fmax(fmax(fabs(x.x), fabs(x.y)), fmax(fabs(y.x), fabs(y.y)));
    const int ex = -__builtin_amdgcn_frexp_exp(big);       // 0 for a big of 0, Inf or NaN
    x = mk(ldexp(x.x, ex), ldexp(x.y, ex));
    y = mk(ldexp(y.x, ex), ldexp(y.y, ex));
    const double xs = abs2(x), ys = abs2(y);
    const double r1 = xs == 0.0 ? 0.0 : rsqrt(xs), r2 = rsqrt(xs + ys);
    c = ys == 0.0 ? 1.0 : xs * r1 * r2;
    s = ys == 0.0 ? czero<double>() : (xs == 0.0 ? conj(y) * r2 : x * conj(y) * (r1 * r2));
  }
}

struct Rot { double c; zd s; };

// b when p, else a, by components (a ternary of structures selects between
// addresses and sends both to scratch memory).
__device__ inline zd sel(bool p, zd b, zd a) { return mk(p ? b.x : a.x, p ? b.y : a.y); }

// a <- a R over columns (k, k + 1) for the rotation list r[k], k = k0 .. hi - 1
// ascending (UP; k0 >= lo may differ from lane to lane) or k = hi - 1 .. lo
// descending, on the row whose entry of column k is a[k ld].  Entries and
// rotations are read four steps ahead.
template <bool UP>
__device__ inline void rotate_row(zd *a, int ld, const Rot *r, int lo, int hi, int k0) {
  zd p = a[(size_t)(UP ? k0 : hi) * ld];
  for (int b = 0; b < hi - lo; b += 4) {
    zd q[4];
    Rot g[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = UP ? min(lo + b + u, hi - 1) : max(hi - 1 - b - u, lo);
      q[u] = a[(size_t)(UP ? k + 1 : k) * ld];
      g[u] = r[k];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = UP ? lo + b + u : hi - 1 - b - u;
      const double c = g[u].c;
      const zd s = g[u].s;
      if (UP) {
        if (k >= k0 && k < hi) {
          a[(size_t)k * ld] = p * c + conj(s) * q[u];
          p = q[u] * c - s * p;
        }
      } else if (k >= lo) {            // p carries the column that moves left
        a[(size_t)(k + 1) * ld] = p * c - s * q[u];
        p = q[u] * c + conj(s) * p;
      }
    }
  }
  a[(size_t)(UP ? hi : lo) * ld] = p;
}

// sum_i conj(v_i) a[i ld] (CONJ) or sum_i a[i ld] v_i over i0 <= i < i1, four
// entries' loads at a time.
template <bool CONJ>
__device__ inline zd strided_dot(const zd *a, int ld, const zd *v, int i0, int i1) {
  zd s[2] = {czero<double>(), czero<double>()};
  for (int i = i0; i < i1; i += 4) {
    zd x[4], w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = min(i + u, i1 - 1);
      x[u] = a[j * ld];
      w[u] = v[j];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u < i1) s[u & 1] = CONJ ? cfmac(s[u & 1], w[u], x[u]) : cfma(s[u & 1], x[u], w[u]);
  }
  return s[0] + s[1];
}
// a[i ld] -= s conj(v_i) (CONJ) or s v_i.
template <bool CONJ>
__device__ inline void strided_sub(zd *a, int ld, const zd *v, zd s, int i0, int i1) {
  for (int i = i0; i < i1; i += 4) {
    zd x[4], w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = min(i + u, i1 - 1);
      x[u] = a[j * ld];
      w[u] = v[j];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (i + u < i1) a[(i + u) * ld] = cfms(x[u], s, CONJ ? conj(w[u]) : w[u]);
  }
}

// LDS of k_schur: H (rows padded by one entry: lane i reading row i meets
// distinct banks), Q column-major, two rotation lists (the Householder vector
// and the triangular eigenvectors of the first nev use their space).
__host__ __device__ inline size_t schur_lds_bytes(int m, int nevmax) {
  const size_t work = sizeof(Rot) * 2 * m, zz = sizeof(zd) * nevmax * nevmax;
  return sizeof(zd) * ((size_t)m * (m + 1) + (size_t)m * m) + (work > zz ? work : zz);
}

__global__ __launch_bounds__(128) void k_schur(const PointDev *__restrict__ pts, zd *__restrict__ small,
                                               KSState *__restrict__ st, int m, int keep, double tol) {
  extern __shared__ zd sl[];
  const PointDev &P = pts[blockIdx.x];
  KSState S = st[blockIdx.x];
  if (S.done) return;
  const int LD = m + 1;
  zd *Hs = sl, *Qs = Hs + m * LD;               // H(i, j) at Hs[i LD + j], Q(i, j) at Qs[j m + i]
  Rot *rot = (Rot *)(Qs + m * m);               // list b at rot + b m
  zd *v = (zd *)rot, *zz = (zd *)rot;
  __shared__ int s_lo[2], s_hi[2];              // range of each list; s_hi < 0 ends a stage
  __shared__ double s_est[KS_NEVMAX];
  zd *Hg = small + P.small_off + SM_H;
  zd *Qg = small + P.small_off + SM_Q;
  zd *Yg = small + P.small_off + SM_Y;
  zd *THg = small + P.small_off + SM_TH;
  const int ldh = KS_MMAX + 1, t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nev = P.nev;
  for (int e = t; e < m * m; e += 128) {
    const int i = e % m, j = e / m;
    Hs[i * LD + j] = Hg[(size_t)j * ldh + i];
    Qs[j * m + i] = (i == j) ? mk(1.0, 0.0) : czero<double>();
  }
  const zd hlast = Hg[(size_t)(m - 1) * ldh + m];
  __syncthreads();
  // --- Householder reduction to Hessenberg form: v = x - alpha e1 with
  // |v|^2 = 2 nx (nx + |x0|).  Both waves form the norms of column k.
  for (int k = 0; k < m - 2; ++k) {
    const int len = m - k - 1;
    const zd xi = (lane < len) ? Hs[(k + 1 + lane) * LD + k] : czero<double>();
    const double nx2 = wave_sum(abs2(xi));
    const zd x0 = lane_get(xi, 0);
    const double below = nx2 - abs2(x0);
    if (below <= 1e-300 * (nx2 + 1e-300)) continue;     // already reduced (the same in every lane)
    const double nx = sqrt(nx2), ax0 = sqrt(abs2(x0));
    const zd ph = (ax0 > 0.0) ? x0 * (1.0 / ax0) : mk(1.0, 0.0);
    const double iv = rsqrt(2.0 * nx * (nx + ax0));
    if (wv == 0 && lane < len) v[lane] = sel(lane == 0, x0 + ph * nx, xi) * iv;
    __syncthreads();
    // H <- (I - 2 v v^H) H on rows k+1.., columns k..m-1: a wave takes 32
    // columns, half a wave each half of the rows
    {
      const int c = k + 32 * wv + (lane & 31), half = lane >> 5, mid = (len + 1) / 2;
      const int i0 = half ? mid : 0, i1 = half ? len : mid;
      zd *col = Hs + (k + 1) * LD + min(c, m - 1);
      zd s = strided_dot<true>(col, LD, v, i0, i1);
      s.x += __shfl_xor(s.x, 32);
      s.y += __shfl_xor(s.y, 32);
      if (c < m) strided_sub<false>(col, LD, v, s * 2.0, i0, i1);
    }
    __syncthreads();
    // H <- H (I - 2 v v^H) on columns k+1.. (wave 0, a row per lane), Q
    // likewise (wave 1)
    if (lane < m) {
      zd *row = wv ? Qs + (size_t)(k + 1) * m + lane : Hs + lane * LD + k + 1;
      const int ld = wv ? m : 1;
      const zd s = strided_dot<false>(row, ld, v, 0, len);
      strided_sub<true>(row, ld, v, s * 2.0, 0, len);
    }
    if (wv == 0) {
      wave_lds_fence();
      if (lane >= 1 && lane < len) Hs[(k + 1 + lane) * LD + k] = czero<double>();
    }
    __syncthreads();
  }
  // --- complex QR sweeps to Schur form (full T and Q); pass n fills list n & 1
  const double eps = 2.220446049250313e-16;
  if (wv == 0) {
    int hi = m - 1, iter = 0, total = 0, n = 0;
    while (hi > 0 && total < 60 * m) {
      // negligible subdiagonals of the active part, all at once
      bool neg = false;
      if (lane >= 1 && lane <= hi) {
        const double sub = cabs1(Hs[lane * LD + lane - 1]);
        const double dia = cabs1(Hs[lane * LD + lane]) + cabs1(Hs[(lane - 1) * LD + lane - 1]);
        neg = sub <= eps * dia || sub < 1e-300;
      }
      const unsigned long long negm = __ballot(neg);
      while (hi > 0 && ((negm >> hi) & 1ull)) {
        if (lane == 0) Hs[hi * LD + hi - 1] = czero<double>();
        --hi;
        iter = 0;
      }
      if (hi == 0) break;
      const unsigned long long below = negm & ((1ull << hi) - 1ull);
      const int lo = below ? 63 - __builtin_clzll(below) : 0;
      if (lo > 0 && lane == 0) Hs[lo * LD + lo - 1] = czero<double>();
      wave_lds_fence();
      ++iter;
      ++total;
      zd mu;
      const zd a = Hs[(hi - 1) * LD + hi - 1], b = Hs[(hi - 1) * LD + hi], c = Hs[hi * LD + hi - 1], d = Hs[hi * LD + hi];
      if (iter % 11 == 10) {
        mu = d + mk(0.75 * sqrt(abs2(c)), 0.0);
      } else {
        const zd half = (a - d) * 0.5;
        const zd disc = half * half + b * c;
        const double r = sqrt(abs2(disc)), sr = sqrt(0.5 * (r + fabs(disc.x)));
        zd sq;
        if (sr == 0.0) sq = czero<double>();
        else if (disc.x >= 0) sq = mk(sr, disc.y / (2.0 * sr));
        else sq = mk(fabs(disc.y) / (2.0 * sr), disc.y >= 0 ? sr : -sr);
        const zd m1 = (a + d) * 0.5 + sq, m2 = (a + d) * 0.5 - sq;
        mu = (abs2(m1 - d) < abs2(m2 - d)) ? m1 : m2;
      }
      // phase 1, lane j = column j.  At rotation k (rows k, k + 1): e = row k,
      // h = row k + 1, hn = row k + 2, hnn = row k + 3 of the lane's column.
      // Columns > k have met no column rotation yet; those of columns k - 1
      // and k are applied to e and h of lanes k - 1 and k as they are found,
      // so one row rotation serves every lane.  (x, y) = e, h of lane k - 1.
      Rot *rl = rot + (n & 1) * m;
      const int col = min(lane, m - 1);
      zd e = Hs[lo * LD + col], h = Hs[(lo + 1) * LD + col], hn = Hs[min(lo + 2, hi) * LD + col];
      zd x = lane_get(e, lo) - mu, y = lane_get(h, lo);
      for (int k = lo; k < hi; ++k) {
        const zd hnn = Hs[min(k + 3, hi) * LD + col];     // past hi: not used
        const zd G = lane_get(hn, k + 1);
        double cg;
        zd sg;
        givens(x, y, cg, sg);
        const zd sc = conj(sg);
        if (lane == 0) { rl[k].c = cg; rl[k].s = sg; }
        const zd f = e * cg + sg * h;
        e = h * cg - sc * e;
        if (lane < m && lane >= (k > lo ? k - 1 : k)) Hs[k * LD + lane] = f;
        // the column rotation (k, k + 1) on rows k + 1 and k + 2
        const zd C1 = lane_get(e, k), D1 = lane_get(e, k + 1);
        x = C1 * cg + sc * D1;
        y = sc * G;
        e = sel(lane == k, x, sel(lane == k + 1, D1 * cg - sg * C1, e));
        h = sel(lane == k, y, sel(lane == k + 1, G * cg, hn));
        hn = hnn;
      }
      if (lane < m && lane >= hi - 1) Hs[hi * LD + lane] = e;
      wave_lds_fence();
      // phase 2, lane i = row i: the sweep's column rotations from max(lo, i) on
      // (those before met row i inside the window)
      if (lane < hi) rotate_row<true>(Hs + lane * LD, 1, rl, lo, hi, max(lo, lane));
      wave_lds_fence();
      if (lane == 0) { s_lo[n & 1] = lo; s_hi[n & 1] = hi; }
      ++n;
      __syncthreads();       // list n - 1 is complete; wave 1 is done with the other one
    }
    if (lane == 0) s_hi[n & 1] = -1;
    __syncthreads();
  } else {
    for (int n = 0;; ++n) {
      __syncthreads();
      const int lo = s_lo[n & 1], hi = s_hi[n & 1];
      if (hi < 0) break;
      if (lane < m) rotate_row<true>(Qs + lane, m, rot + (n & 1) * m, lo, hi, lo);
    }
  }
  __syncthreads();
  // --- reorder: bring the `keep` eigenvalues of largest modulus to the front;
  // pass pos fills list pos & 1 (an empty range when nothing moves)
  if (wv == 0) {
    for (int pos = 0; pos < keep; ++pos) {
      const double av = (lane >= pos && lane < m) ? sqrt(abs2(Hs[min(lane, m - 1) * LD + min(lane, m - 1)])) : -1.0;
      double bv = av;
      for (int off = 32; off > 0; off >>= 1) bv = fmax(bv, __shfl_xor(bv, off));
      const int best = schur_pick(__ballot(av == bv), pos, m);      // a row of H whatever its entries
      Rot *rl = rot + (pos & 1) * m;
      const zd t22 = Hs[best * LD + best];                          // the eigenvalue that moves up
      for (int k = best - 1; k >= pos; --k) {
        const zd t11 = Hs[k * LD + k];
        double cg;
        zd sg;
        givens(Hs[k * LD + k + 1], t22 - t11, cg, sg);
        if (lane == 0) { rl[k].c = cg; rl[k].s = sg; }
        const int jj = k + lane;
        if (jj < m) {
          const zd p = Hs[k * LD + jj], q = Hs[(k + 1) * LD + jj];
          Hs[k * LD + jj] = p * cg + sg * q;
          Hs[(k + 1) * LD + jj] = q * cg - conj(sg) * p;
        }
        wave_lds_fence();
        if (lane <= k + 1) {
          const zd p = Hs[lane * LD + k], q = Hs[lane * LD + k + 1];
          // rows k and k + 1 of the 2 x 2 block are known: [t22, .; 0, t11]
          Hs[lane * LD + k] = sel(lane == k, t22, sel(lane == k + 1, czero<double>(), p * cg + conj(sg) * q));
          Hs[lane * LD + k + 1] = sel(lane == k + 1, t11, q * cg - sg * p);
        }
        wave_lds_fence();
      }
      if (lane == 0) { s_lo[pos & 1] = pos; s_hi[pos & 1] = best; }
      __syncthreads();
    }
  } else {
    for (int pos = 0; pos < keep; ++pos) {
      __syncthreads();
      if (lane < m && s_hi[pos & 1] > pos) rotate_row<false>(Qs + lane, m, rot + (pos & 1) * m, pos, s_hi[pos & 1], 0);
    }
  }
  __syncthreads();
  // --- eigenvectors of T for the first nev (thread i handles pair i; entries
  // past i vanish)
  if (t < nev) {
    const int i = t;
    zd *z = zz + i * nev;
    const zd ti = Hs[i * LD + i];
    const double smin = fmax(eps * cabs(ti), 1e-300);
    z[i] = mk(1.0, 0.0);
    for (int l = i - 1; l >= 0; --l) {
      zd s = czero<double>();
      for (int c = l + 1; c <= i; ++c) s = cfma(s, Hs[l * LD + c], z[c]);
      zd d = Hs[l * LD + l] - ti;
      if (cabs(d) < smin) d = mk(smin, 0.0);
      z[l] = czero<double>() - cdiv(s, d);
    }
  }
  __syncthreads();
  // y_i = Q z_i, normalised (a wave per pair, a row per lane); residual
  // estimate |h_{m,m-1}| |y_i[m-1]|
  for (int i = wv; i < nev; i += 2) {
    const zd *z = zz + i * nev;
    zd s = czero<double>();
    if (lane < m)
      for (int c = 0; c <= i; ++c) s = cfma(s, Qs[c * m + lane], z[c]);
    const double inv = 1.0 / sqrt(wave_sum(abs2(s)));
    if (lane < m) Yg[(size_t)i * KS_MMAX + lane] = s * inv;
    if (lane == m - 1) s_est[i] = cabs(hlast) * cabs(s) * inv / fmax(cabs(Hs[i * LD + i]), 1e-300);
  }
  // write Q (the kept columns), theta and T
  for (int e = t; e < m * keep; e += 128) {
    const int i = e % m, j = e / m;
    Qg[(size_t)j * KS_MMAX + i] = Qs[j * m + i];
  }
  for (int i = t; i < m; i += 128) THg[i] = Hs[i * LD + i];
  for (int e = t; e < keep * keep; e += 128) {
    const int i = e % keep, j = e / keep;
    Hg[(size_t)j * ldh + i] = (i <= j) ? Hs[i * LD + j] : czero<double>();
  }
  __syncthreads();
  if (t == 0) {
    const double mx = est_max(s_est, nev);
    S.resmax = mx;
    S.cycles += 1;
    if (S.cycles == 1 || mx < 0.1 * S.best) { S.best = fmin(mx, S.cycles == 1 ? mx : S.best); S.stall = 0; }
    else S.stall += 1;
    S.best = fmin(S.best, mx);
    // converged; else stop this point on NaN (the factors of a singular matrix:
    // nothing left to iterate) or without tenfold progress in three cycles (an
    // ill-conditioned cluster among the wanted pairs)
    S.done = (mx <= tol) ? 1 : ((mx != mx || S.stall >= 3) ? 2 : 0);
    st[blockIdx.x] = S;
  }
}

// ---------------------------------------------------------------------------
// The same on one wave, rotation by rotation in LDS, for mode tracking only
// (Gram-Schmidt by groups of four columns, GS4 of k_arnoldi, goes with it).
// Tracking feeds the eigenvalue of one step into the shift of the next, and a
// point whose residual floor lies at the acceptance limit of the inverse
// iteration (1e-14) changes its info code with the last bits of that shift:
// with the sums of k_schur in the fallback, 1 of 25 tracked batches returned
// other codes.  So the fallback of a tracked point keeps this order of
// operations; it is rare (a quarter of 16-curve batches have such a point).
// It costs such a point 2.95 ms a cycle (m = 40) where k_schur takes 1.21, and
// 37 us a Gram-Schmidt step (n = 480) where the other form takes 14.
// ---------------------------------------------------------------------------
__device__ inline void givens_seq(zd x, zd y, double &c, zd &s) {
  const double ax = cabs(x), ay = cabs(y);
  if (ay == 0.0) { c = 1.0; s = czero<double>(); return; }
  if (ax == 0.0) { c = 0.0; s = conj(y) * (1.0 / ay); return; }
  const double r = hypot(ax, ay);
  c = ax / r;
  s = (x * (1.0 / ax)) * conj(y) * (1.0 / r);
}

__global__ __launch_bounds__(64) void k_schur_seq(const PointDev *__restrict__ pts, zd *__restrict__ small,
                                              KSState *__restrict__ st, int m, int keep, double tol) {
  extern __shared__ zd sl[];
  const PointDev &P = pts[blockIdx.x];
  KSState S = st[blockIdx.x];
  if (S.done) return;
  zd *Hs = sl, *Q = Hs + m * m, *v = Q + m * m, *zz = v + m;   // zz: KS_NEVMAX * m
  zd *Hg = small + P.small_off + SM_H;
  zd *Qg = small + P.small_off + SM_Q;
  zd *Yg = small + P.small_off + SM_Y;
  zd *THg = small + P.small_off + SM_TH;
  const int ldh = KS_MMAX + 1, t = threadIdx.x;
  const int nev = P.nev;
  for (int e = t; e < m * m; e += 64) {
    const int i = e % m, j = e / m;
    Hs[i * m + j] = Hg[(size_t)j * ldh + i];   // row-major in LDS
    Q[i * m + j] = (i == j) ? mk(1.0, 0.0) : czero<double>();
  }
  const zd hlast = Hg[(size_t)(m - 1) * ldh + m];
  __syncthreads();
  // --- Householder reduction to Hessenberg form
  for (int k = 0; k < m - 2; ++k) {
    const int len = m - k - 1;
    double nx = 0.0;
    for (int i = 0; i < len; ++i) nx += abs2(Hs[(k + 1 + i) * m + k]);
    double below = nx - abs2(Hs[(k + 1) * m + k]);
    if (below <= 1e-300 * (nx + 1e-300)) continue;     // already reduced
    nx = sqrt(nx);
    const zd x0 = Hs[(k + 1) * m + k];
    const double ax0 = cabs(x0);
    const zd ph = (ax0 > 0.0) ? x0 * (1.0 / ax0) : mk(1.0, 0.0);
    const zd alpha = ph * (-nx);
    // v = x - alpha e1, normalised
    for (int i = t; i < len; i += 64) v[i] = (i == 0) ? x0 - alpha : Hs[(k + 1 + i) * m + k];
    __syncthreads();
    double vn = 0.0;
    for (int i = 0; i < len; ++i) vn += abs2(v[i]);
    vn = sqrt(vn);
    __syncthreads();
    for (int i = t; i < len; i += 64) v[i] = v[i] * (1.0 / vn);
    __syncthreads();
    // H <- (I - 2 v v^H) H  on rows k+1.., columns k..m-1
    for (int c = k + t; c < m; c += 64) {
      zd s = czero<double>();
      for (int i = 0; i < len; ++i) s = cfmac(s, v[i], Hs[(k + 1 + i) * m + c]);
      for (int i = 0; i < len; ++i) Hs[(k + 1 + i) * m + c] = cfms(Hs[(k + 1 + i) * m + c], v[i], s * 2.0);
    }
    __syncthreads();
    // H <- H (I - 2 v v^H) on columns k+1.., all rows; Q likewise
    for (int rr = t; rr < 2 * m; rr += 64) {
      zd *row = (rr < m) ? &Hs[rr * m] : &Q[(rr - m) * m];
      zd s = czero<double>();
      for (int i = 0; i < len; ++i) s = cfma(s, row[k + 1 + i], v[i]);
      for (int i = 0; i < len; ++i) row[k + 1 + i] = cfms(row[k + 1 + i], s * 2.0, conj(v[i]));
    }
    __syncthreads();
    if (t == 0)
      for (int i = 2; i < len + 1; ++i) Hs[(k + i) * m + k] = czero<double>();
    __syncthreads();
  }
  // --- complex QR iterations to Schur form (full T and Q)
  const double eps = 2.220446049250313e-16;
  int hi = m - 1, iter = 0, total = 0;
  while (hi > 0 && total < 60 * m) {
    int lo = hi;
    while (lo > 0) {
      const double sub = cabs1(Hs[lo * m + lo - 1]);
      const double dia = cabs1(Hs[lo * m + lo]) + cabs1(Hs[(lo - 1) * m + lo - 1]);
      if (sub <= eps * dia || sub < 1e-300) break;
      --lo;
    }
    if (lo > 0) {
      __syncthreads();
      if (t == 0) Hs[lo * m + lo - 1] = czero<double>();
      __syncthreads();
    }
    if (lo == hi) { --hi; iter = 0; continue; }
    ++iter; ++total;
    zd mu;
    const zd a = Hs[(hi - 1) * m + hi - 1], b = Hs[(hi - 1) * m + hi], c = Hs[hi * m + hi - 1], d = Hs[hi * m + hi];
    if (iter % 11 == 10) {
      mu = d + mk(0.75 * cabs(c), 0.0);
    } else {
      const zd half = (a - d) * 0.5;
      zd disc = half * half + b * c;
      // complex sqrt
      const double r = cabs(disc);
      double sr = sqrt(0.5 * (r + fabs(disc.x)));
      zd sq;
      if (sr == 0.0) sq = czero<double>();
      else if (disc.x >= 0) sq = mk(sr, disc.y / (2.0 * sr));
      else sq = mk(fabs(disc.y) / (2.0 * sr), disc.y >= 0 ? sr : -sr);
      const zd m1 = (a + d) * 0.5 + sq, m2 = (a + d) * 0.5 - sq;
      mu = (cabs(m1 - d) < cabs(m2 - d)) ? m1 : m2;
    }
    for (int k = lo; k < hi; ++k) {
      zd x, y;
      if (k == lo) { x = Hs[lo * m + lo] - mu; y = Hs[(lo + 1) * m + lo]; }
      else { x = Hs[k * m + k - 1]; y = Hs[(k + 1) * m + k - 1]; }
      double cg; zd sg;
      givens_seq(x, y, cg, sg);
      __syncthreads();
      const int c0 = (k > lo) ? k - 1 : lo;
      for (int jj = c0 + t; jj < m; jj += 64) {
        const zd p = Hs[k * m + jj], q = Hs[(k + 1) * m + jj];
        Hs[k * m + jj] = p * cg + sg * q;
        Hs[(k + 1) * m + jj] = q * cg - conj(sg) * p;
      }
      __syncthreads();
      const int rmax = min(k + 2, hi);
      for (int ii = t; ii <= rmax; ii += 64) {
        const zd p = Hs[ii * m + k], q = Hs[ii * m + k + 1];
        Hs[ii * m + k] = p * cg + conj(sg) * q;
        Hs[ii * m + k + 1] = q * cg - sg * p;
      }
      for (int ii = t; ii < m; ii += 64) {
        const zd p = Q[ii * m + k], q = Q[ii * m + k + 1];
        Q[ii * m + k] = p * cg + conj(sg) * q;
        Q[ii * m + k + 1] = q * cg - sg * p;
      }
      __syncthreads();
      if (k > lo && t == 0) Hs[(k + 1) * m + k - 1] = czero<double>();
      __syncthreads();
    }
  }
  __syncthreads();
  // --- reorder: bring the `keep` eigenvalues of largest modulus to the front
  for (int pos = 0; pos < keep; ++pos) {
    int best = pos;
    double bv = cabs(Hs[pos * m + pos]);
    for (int i = pos + 1; i < m; ++i) {
      const double vv = cabs(Hs[i * m + i]);
      if (vv > bv) { bv = vv; best = i; }
    }
    for (int k = best - 1; k >= pos; --k) {
      const zd t11 = Hs[k * m + k], t22 = Hs[(k + 1) * m + k + 1];
      double cg; zd sg;
      givens_seq(Hs[k * m + k + 1], t22 - t11, cg, sg);
      __syncthreads();
      for (int jj = k + t; jj < m; jj += 64) {
        const zd p = Hs[k * m + jj], q = Hs[(k + 1) * m + jj];
        Hs[k * m + jj] = p * cg + sg * q;
        Hs[(k + 1) * m + jj] = q * cg - conj(sg) * p;
      }
      __syncthreads();
      for (int ii = t; ii <= k + 1; ii += 64) {
        const zd p = Hs[ii * m + k], q = Hs[ii * m + k + 1];
        Hs[ii * m + k] = p * cg + conj(sg) * q;
        Hs[ii * m + k + 1] = q * cg - sg * p;
      }
      for (int ii = t; ii < m; ii += 64) {
        const zd p = Q[ii * m + k], q = Q[ii * m + k + 1];
        Q[ii * m + k] = p * cg + conj(sg) * q;
        Q[ii * m + k + 1] = q * cg - sg * p;
      }
      __syncthreads();
      if (t == 0) {
        Hs[k * m + k] = t22;
        Hs[(k + 1) * m + k + 1] = t11;
        Hs[(k + 1) * m + k] = czero<double>();
      }
      __syncthreads();
    }
  }
  // --- eigenvectors of T for the first nev (lane i handles pair i)
  if (t < nev) {
    const int i = t;
    zd *z = zz + i * m;
    const zd ti = Hs[i * m + i];
    const double smin = fmax(eps * cabs(ti), 1e-300);
    for (int l = 0; l < m; ++l) z[l] = czero<double>();
    z[i] = mk(1.0, 0.0);
    for (int l = i - 1; l >= 0; --l) {
      zd s = czero<double>();
      for (int c = l + 1; c <= i; ++c) s = cfma(s, Hs[l * m + c], z[c]);
      zd d = Hs[l * m + l] - ti;
      if (cabs(d) < smin) d = mk(smin, 0.0);
      z[l] = czero<double>() - cdiv(s, d);
    }
  }
  __syncthreads();
  // y_i = Q z_i, normalised; residual estimate |h_{m,m-1}| |y_i[m-1]|
  __shared__ double s_est[KS_NEVMAX];
  if (t < nev) {
    const int i = t;
    const zd *z = zz + i * m;
    double nn = 0.0;
    zd ylast = czero<double>();
    for (int r = 0; r < m; ++r) {
      zd s = czero<double>();
      for (int c = 0; c <= i; ++c) s = cfma(s, Q[r * m + c], z[c]);
      nn += abs2(s);
      if (r == m - 1) ylast = s;
    }
    const double inv = 1.0 / sqrt(nn);
    for (int r = 0; r < m; ++r) {
      zd s = czero<double>();
      for (int c = 0; c <= i; ++c) s = cfma(s, Q[r * m + c], z[c]);
      Yg[(size_t)i * KS_MMAX + r] = s * inv;
    }
    const zd th = Hs[i * m + i];
    s_est[i] = cabs(hlast) * cabs(ylast) * inv / fmax(cabs(th), 1e-300);
  }
  __syncthreads();
  // write T (row-major -> column-major global H) and Q, theta
  for (int e = t; e < m * m; e += 64) {
    const int i = e % m, j = e / m;
    Qg[(size_t)j * KS_MMAX + i] = Q[i * m + j];
  }
  for (int i = t; i < m; i += 64) THg[i] = Hs[i * m + i];
  for (int e = t; e < keep * keep; e += 64) {
    const int i = e % keep, j = e / keep;
    Hg[(size_t)j * ldh + i] = (i <= j) ? Hs[i * m + j] : czero<double>();
  }
  __syncthreads();
  if (t == 0) {
    const double mx = est_max(s_est, nev);
    S.resmax = mx;
    S.cycles += 1;
    if (S.cycles == 1 || mx < 0.1 * S.best) { S.best = fmin(mx, S.cycles == 1 ? mx : S.best); S.stall = 0; }
    else S.stall += 1;
    S.best = fmin(S.best, mx);
    // converged; else stop this point on NaN (the factors of a singular matrix:
    // nothing left to iterate) or without tenfold progress in three cycles (an
    // ill-conditioned cluster among the wanted pairs)
    S.done = (mx <= tol) ? 1 : ((mx != mx || S.stall >= 3) ? 2 : 0);
    st[blockIdx.x] = S;
  }
}

// Krylov-Schur truncation to `keep` columns: V <- V Q(:, 0:keep), v_keep <- v_m,
// H <- [T_keep; b^H], b^H = h_{m,m-1} Q(m-1, 0:keep).
template <int NT, int KMAX>
__global__ __launch_bounds__(NT) void k_restart(const PointDev *__restrict__ pts, zd *__restrict__ Vall,
                                                zd *__restrict__ small, KSState *__restrict__ st, int m, int keep) {
  // grid: x = points, y = chunks of NT rows; the first chunk's work-group also
  // rebuilds H (the others read only V and Q)
  const PointDev &P = pts[blockIdx.x];
  KSState S = st[blockIdx.x];
  if (S.done || (int)blockIdx.y * NT >= P.nvec) return;
  __shared__ zd s_q[KS_MMAX * KMAX];
  const int t = threadIdx.x, nv = P.nvec;
  const size_t ldv = (size_t)nv;
  zd *V = Vall + P.vec_off;
  zd *H = small + P.small_off + SM_H;
  const zd *Qg = small + P.small_off + SM_Q;
  const int ldh = KS_MMAX + 1;
  for (int e = t; e < m * keep; e += NT) {
    const int r = e % m, c = e / m;
    s_q[r * KMAX + c] = Qg[(size_t)c * KS_MMAX + r];
  }
  const zd hlast = H[(size_t)(m - 1) * ldh + m];
  __syncthreads();
  if (const int r = blockIdx.y * NT + t; r < nv) {
    zd acc[KMAX];
#pragma unroll
    for (int c = 0; c < KMAX; ++c) acc[c] = czero<double>();
    for_loaded<4>(m, [&](int l) { return V[(size_t)l * ldv + r]; }, [&](int l, zd v) {
#pragma unroll
      for (int c = 0; c < KMAX; ++c)
        if (c < keep) acc[c] = cfma(acc[c], v, s_q[l * KMAX + c]);
    });
    const zd vm = V[(size_t)m * ldv + r];
#pragma unroll
    for (int c = 0; c < KMAX; ++c)
      if (c < keep) V[(size_t)c * ldv + r] = acc[c];
    V[(size_t)keep * ldv + r] = vm;
  }
  if (blockIdx.y) return;
  __syncthreads();
  // rebuild H: T block already written by k_schur in rows/cols < keep
  for (int e = t; e < ldh * KS_MMAX; e += NT) {
    const int i = e % ldh, j = e / ldh;
    if (j >= keep || i > keep) H[e] = czero<double>();
  }
  __syncthreads();
  // b^T = h_{m,m-1} e_{m-1}^T Q(:, 0:keep)
  for (int j = t; j < keep; j += NT) H[(size_t)j * ldh + keep] = hlast * s_q[(m - 1) * KMAX + j];
  if (t == 0) { S.j0 = keep; S.k = keep; st[blockIdx.x] = S; }
}

// Final Ritz pairs: x_i = V y_i, omega_i = sigma + 1/theta_i, getevec-style
// normalisation (first entry of largest modulus among the first 5 ny
// components becomes 1, getevec.f90:179-189), FP64 relative residual.
// Whether node i lies in the farfield: the outer eighth of the Chebyshev
// nodes (node 0 .. ceil(ny/8) - 1, eta near 1); for a finite-difference
// point, whose node 0 is the wall, the nodes of the outer half of the domain,
// y >= ymax/2, with y formed as k_nodes forms it (for yi = 2/46, ymax = 50
// the Chebyshev window starts at y = 25.7 too).
__device__ inline bool farfield_node(const PointDev &P, int i) {
  if (!P.fd) return i < (P.ny + 7) / 8;
  const double dy = 1.0 / (double)(P.ny - 1);
  const double aa = P.ymax * P.yi / (P.ymax - 2.0 * P.yi), bb = 1.0 + aa / P.ymax;
  const double eta = (double)i * dy;
  return aa * eta / (bb - eta) >= 0.5 * P.ymax;
}

// Largest modulus over the farfield nodes (all five variables) of a vector
// normalised to a largest entry of modulus 1.  Discrete modes decay there,
// the continuous spectrum does not.
template <int NT>
__device__ double farfield_ratio(const PointDev &P, const zd *x, zd *red) {
  double a = 0.0, b = 0.0;
  for (int r = threadIdx.x; r < P.n; r += NT) {
    const double v = abs2(x[r]);
    b = fmax(b, v);
    if (farfield_node(P, r / 5)) a = fmax(a, v);
  }
  for (int off = 32; off > 0; off >>= 1) {
    a = fmax(a, __shfl_xor(a, off));
    b = fmax(b, __shfl_xor(b, off));
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) { red[threadIdx.x >> 6] = mk(a, b); }
  __syncthreads();
  for (int w = 0; w < NT / 64; ++w) { a = fmax(a, red[w].x); b = fmax(b, red[w].y); }
  __syncthreads();
  return b > 0.0 ? sqrt(a / b) : 1.0;
}

template <int NT>
__global__ __launch_bounds__(NT) void k_final(const PointDev *__restrict__ pts, const zd *__restrict__ Vall,
                                              const zd *__restrict__ small, const zd *__restrict__ coef,
                                              const double *__restrict__ ops, const double *__restrict__ norms,
                                              int m, zd *__restrict__ eval, zd *__restrict__ evec,
                                              double *__restrict__ resid, double *__restrict__ ffo, int npadmax,
                                              int nymax, int nvecmax) {
  extern __shared__ zd lds[];
  const PointDev &P = pts[blockIdx.x];
  OpLds L(lds, NT, npadmax, nymax, 1, nvecmax);
  const int t = threadIdx.x, nv = P.nvec, n = P.n;
  const size_t ldv = (size_t)nv;
  const zd *V = Vall + P.vec_off;
  const zd *Yg = small + P.small_off + SM_Y;
  const zd *THg = small + P.small_off + SM_TH;
  zd *out = evec + P.out_off;
  for (int i = 0; i < P.nev; ++i) {
    const zd th = THg[i];
    const zd om = P.shift + cdiv(mk(1.0, 0.0), th);
    for (int r = t; r < nv; r += NT) {
      zd s = czero<double>();
      for_loaded<8>(m, [&](int l) { return V[(size_t)l * ldv + r]; },
                    [&](int l, zd v) { s = cfma(s, v, Yg[(size_t)i * KS_MMAX + l]); });
      L.z[r] = s;
    }
    __syncthreads();
    // first entry of largest modulus among the first n components
    double bm = -1.0; int bi = 0x7fffffff;
    for (int r = t; r < n; r += NT) { const double a = cabs(L.z[r]); if (a > bm) { bm = a; bi = r; } }
    // all-NaN vector: no entry compares greater
    const zd scale = L.z[clamp_index(block_argmax<NT>(bm, bi, L.red), n)];
    __syncthreads();
    if (scale_ok(scale))
      for (int r = t; r < nv; r += NT) L.z[r] = cdiv(L.z[r], scale);
    __syncthreads();
    {
      const double ff = farfield_ratio<NT>(P, L.z, L.red);
      if (t == 0 && ffo) ffo[(size_t)blockIdx.x * KS_NEVMAX + i] = ff;
    }
    // FP64 residual at the Ritz value and at the Rayleigh-quotient value of the
    // same vector; the smaller one is kept.  An operator error along the wanted
    // eigenvector (the near-null direction of A - sigma B when the shift is
    // close) moves only the Ritz value, not the vector, so the quotient with
    // the exact pencil recovers the eigenvalue.
    double rn, xn, den;
    zd om_out = om;
    if (P.itype == 1) {
      pencil_apply<NT>(P, coef, ops, FORM_AM, P.shift, L.z, L.y, L.X1, L.X2, L.red);
      pencil_apply<NT>(P, coef, ops, FORM_BM, P.shift, L.z, L.rhs, L.X1, L.X2, L.red);
      zd d3[3] = {czero<double>(), czero<double>(), czero<double>()};
      for (int r = red_first(); r < n; r += RT) {
        d3[0] = cfmac(d3[0], L.z[r], L.y[r]);
        d3[1] = cfmac(d3[1], L.z[r], L.rhs[r]);
      }
      block_reduce<NT, 3>(d3, L.red);
      const zd om_rq = (cabs(d3[1]) > 0.0) ? cdiv(d3[0], d3[1]) : om;
      zd part[3] = {czero<double>(), czero<double>(), czero<double>()};
      for (int r = red_first(); r < n; r += RT) {
        part[0].x += abs2(L.y[r] - om * L.rhs[r]);
        part[1].x += abs2(L.y[r] - om_rq * L.rhs[r]);
        part[2].x += abs2(L.z[r]);
      }
      block_reduce<NT, 3>(part, L.red);
      const bool use_rq = part[1].x < part[0].x;
      om_out = use_rq ? om_rq : om;
      rn = sqrt(use_rq ? part[1].x : part[0].x);
      xn = sqrt(part[2].x);
      den = sqrt(norms[blockIdx.x * 4 + 0]) + cabs(om_out) * sqrt(norms[blockIdx.x * 4 + 1]);
    } else {
      // C0 phi -> y, C1 phi -> rhs, C2 phi -> res
      pencil_apply<NT>(P, coef, ops, FORM_C0, P.shift, L.z, L.y, L.X1, L.X2, L.red);
      pencil_apply<NT>(P, coef, ops, FORM_C1, P.shift, L.z, L.rhs, L.X1, L.X2, L.red);
      pencil_apply<NT>(P, coef, ops, FORM_C2, P.shift, L.z, L.res, L.X1, L.X2, L.red);
      zd d3[3] = {czero<double>(), czero<double>(), czero<double>()};
      for (int r = red_first(); r < n; r += RT) {
        d3[0] = cfmac(d3[0], L.z[r], L.y[r]);
        d3[1] = cfmac(d3[1], L.z[r], L.rhs[r]);
        d3[2] = cfmac(d3[2], L.z[r], L.res[r]);
      }
      block_reduce<NT, 3>(d3, L.red);
      // roots of c2 a^2 + c1 a + c0 = 0 nearest the Ritz value
      zd om_rq = om;
      if (cabs(d3[2]) > 0.0) {
        const zd bb = cdiv(d3[1], d3[2] * 2.0), cc = cdiv(d3[0], d3[2]);
        zd disc = bb * bb - cc;
        const double rr = cabs(disc);
        const double sr = sqrt(0.5 * (rr + fabs(disc.x)));
        zd sq;
        if (sr == 0.0) sq = czero<double>();
        else if (disc.x >= 0) sq = mk(sr, disc.y / (2.0 * sr));
        else sq = mk(fabs(disc.y) / (2.0 * sr), disc.y >= 0 ? sr : -sr);
        const zd r1 = czero<double>() - bb + sq, r2 = czero<double>() - bb - sq;
        om_rq = (cabs(r1 - om) < cabs(r2 - om)) ? r1 : r2;
      } else if (cabs(d3[1]) > 0.0) {
        om_rq = czero<double>() - cdiv(d3[0], d3[1]);
      }
      zd part[3] = {czero<double>(), czero<double>(), czero<double>()};
      for (int r = red_first(); r < n; r += RT) {
        part[0].x += abs2(L.y[r] + om * L.rhs[r] + (om * om) * L.res[r]);
        part[1].x += abs2(L.y[r] + om_rq * L.rhs[r] + (om_rq * om_rq) * L.res[r]);
        part[2].x += abs2(L.z[r]);
      }
      block_reduce<NT, 3>(part, L.red);
      const bool use_rq = part[1].x < part[0].x;
      om_out = use_rq ? om_rq : om;
      rn = sqrt(use_rq ? part[1].x : part[0].x);
      xn = sqrt(part[2].x);
      const double a = cabs(om_out);
      den = sqrt(norms[blockIdx.x * 4 + 0]) + a * sqrt(norms[blockIdx.x * 4 + 1]) + a * a * sqrt(norms[blockIdx.x * 4 + 2]);
    }
    if (t == 0) {
      eval[(size_t)blockIdx.x * KS_NEVMAX + i] = om_out;
      resid[(size_t)blockIdx.x * KS_NEVMAX + i] = rn / (den * xn);
    }
    for (int r = t; r < nv; r += NT) out[(size_t)i * nv + r] = L.z[r];
    __syncthreads();
  }
}

// One shifted solve M x = b (factors from k_lu, `ir` refinement steps); used by
// the stab_shifted_solve entry point.
template <typename T, int NB, int NT>
__global__ __launch_bounds__(NT) void k_solve_one(const PointDev *__restrict__ pts, const cx<T> *__restrict__ mats,
                                                  const int *__restrict__ pivs, const cx<T> *__restrict__ blks,
                                                  const double *__restrict__ scales, const zd *__restrict__ coef,
                                                  const double *__restrict__ ops, const zd *__restrict__ b,
                                                  zd *__restrict__ x, int ir, int npadmax, int nymax) {
  extern __shared__ zd lds[];
  const PointDev &P = pts[blockIdx.x];
  OpLds L(lds, NT, npadmax, nymax, 1, npadmax);
  const cx<T> *A = mats + P.mat_off;
  const int *ipiv = pivs + P.piv_off;
  const cx<T> *Lb = blks + P.blk_off, *Ub = nullptr;
  const double *dr = scales + P.scale_off, *dc = dr + P.npad;
  for (int r = threadIdx.x; r < P.n; r += NT) L.rhs[r] = b[r];
  __syncthreads();
  shifted_solve<T, NB, NT>(P, A, ipiv, Lb, Ub, dr, dc, coef, ops, ir, L);
  for (int r = threadIdx.x; r < P.n; r += NT) x[r] = L.y[r];
}

// Principal square root of a complex number.
__device__ inline zd zsqrt(zd z) {
  const double r = cabs(z);
  const double sr = sqrt(0.5 * (r + fabs(z.x)));
  if (sr == 0.0) return czero<double>();
  if (z.x >= 0) return mk(sr, z.y / (2.0 * sr));
  return mk(fabs(z.y) / (2.0 * sr), z.y >= 0 ? sr : -sr);
}

// ---------------------------------------------------------------------------
// Two-vector residual inverse iteration with a 2 x 2 Rayleigh-Ritz step, for
// temporal points whose single-vector iteration (k_invit) missed.  There the
// two eigenvalues nearest the shift are nearly equidistant from it, so one
// vector contracts towards neither (or settles on the nearer one when the
// other is wanted); a basis X = [x1, x2] converges to both at the rate
// max |lambda_{1,2} - sigma| / |lambda_3 - sigma| per step:
//   X orthonormal (FP64); projected pencil (X^H A X, X^H B X); its two
//   eigenpairs (theta_k, y_k) from det(A~ - theta B~) = 0; Ritz vectors
//   u_k = X y_k with FP64 residuals r_k = A u_k - theta_k B u_k; new basis
//   x_k = u_k - L(sigma)^-1 r_k.
// Starts from the vector k_invit left in column 0 of the point's block (x1)
// and x2 = L(sigma)^-1 B x1, on the factors k_invit used.  A pair has
// converged when its relative residual is below tol or has not halved for
// three steps while below 1e-12.  The wanted pair (want 0: the least stable
// of the pairs that pass lead2_discrete; want 1: the one nearest the shift)
// is iterated until it has converged and the other pair has converged too, or
// has a residual below 1e-10 and can no longer outrank it (lead2_competes,
// the test the host applies to the results); at most maxit steps.
// Outputs, k = 0, 1: eval2[2 p + k], resid2[2 p + k], ff2[2 p + k] and the
// Ritz vector (getevec normalisation) in column k of p's block;
// iters[p] += solves.  It runs inside k_invit after a point's first pass
// (fused) or as k_invit2 after the whole first pass.
// ---------------------------------------------------------------------------
// The discrete-mode test of the leading-mode selection for temporal points:
// farfield ratio below STAB_FARFIELD_MAX and phase speed off the continuum.
__host__ __device__ inline bool lead2_discrete(double alpha_r, zd ev, double ff) {
  if (!(ff < STAB_FARFIELD_MAX)) return false;
  if (alpha_r == 0.0) return true;
  return fabs(ev.x / alpha_r - 1.0) > STAB_CONTINUUM_BAND;
}

// Whether pair o (residual rel_o, farfield ratio ff_o), not converged, could
// still outrank the converged pair w.  Its eigenvalue error is taken as
// 1e5 rel_o max(|theta_o|, 1e-2) (a relative condition number of 1e5; the
// discrete modes of these pencils stay below it); its farfield ratio is
// trusted once rel_o < 1e-8.
__host__ __device__ inline bool lead2_competes(int want, double alpha_r, zd sigma, zd th_w, zd th_o, double rel_o,
                                               double ff_o) {
  const double err = 1e5 * rel_o * fmax(cabs(th_o), 1e-2);
  if (want == 1) return cabs(th_o - sigma) < cabs(th_w - sigma) + err;
  const bool maybe_discrete = !(rel_o < 1e-8) || lead2_discrete(alpha_r, th_o, ff_o);
  return maybe_discrete && th_o.y > th_w.y - err;
}

// The second pass for point p (P = its descriptor), x1 holding the first
// pass's vector (getevec normalisation) on entry.  x1, x2, a1, a2 and tmp2 (2
// NT entries with 256 threads, 128 with more) are LDS; b1 and b2 may be
// global: the products that write them end in a barrier, and the sums that
// read them, whose stride (RT) is not the work-group's, come after it.  L supplies the solve's scratch (y, rhs, tmp, w2), the
// products' (X1, X2, red) and nothing else, so x1 .. a2 may alias L.z, L.res,
// L.y and L.rhs as long as a1, a2 are not L.rhs, L.y before the first step's
// solve is done (they are written only inside the loop).
// Whether the second pass takes a point after the first (maxit1 steps):
// a temporal point whose LU succeeded and which the first pass left
// unconverged, not discrete (unless want == 1), or converged only after 3/4
// of its steps.  The host applies the same rule to the same data.
__host__ __device__ inline bool lead2_needed(int info, int itype, int flag, int want, double alpha_r, zd ev,
                                             double ff, int iters, int maxit1) {
  if (info != 0 || itype != 1) return false;
  const bool ok1 = flag == 0 && (want == 1 || lead2_discrete(alpha_r, ev, ff));
  return !(ok1 && 4 * iters < 3 * (maxit1 + 1));
}

template <typename T, int NB, int NT>
__device__ __forceinline__ void invit2_point(const PointDev &P, int p, const cx<T> *__restrict__ mats,
                                             const int *__restrict__ pivs, const cx<T> *__restrict__ blks,
                                             const double *__restrict__ scales, const zd *__restrict__ coef,
                                             const double *__restrict__ ops, const double *__restrict__ norms,
                                             int maxit, double tol, int want, zd *__restrict__ eval2,
                                             zd *__restrict__ evec, double *__restrict__ resid2,
                                             double *__restrict__ ff2, int *__restrict__ iters, OpLds &L, zd *x1,
                                             zd *x2, zd *a1, zd *b1, zd *a2, zd *b2, zd *tmp2) {
  const int t = threadIdx.x, n = P.n, nv = P.nvec;
  const cx<T> *A = mats + P.mat_off;
  const int *ipiv = pivs + P.piv_off;
  const cx<T> *Lb = blks + P.blk_off, *Ub = nullptr;
  const double *dr = scales + P.scale_off, *dc = dr + P.npad;
  const double nA = sqrt(norms[p * 4 + 0]), nB = sqrt(norms[p * 4 + 1]);
  const zd sg = P.shift;
  zd *out = evec + P.out_off;
  pencil_apply<NT>(P, coef, ops, FORM_BM, sg, x1, L.rhs, L.X1, L.X2, L.red);
  shifted_solve<T, NB, NT, true>(P, A, ipiv, Lb, Ub, dr, dc, coef, ops, 0, L);
  for (int r = t; r < n; r += NT) x2[r] = L.y[r];
  __syncthreads();
  int nsolve = 1;
  zd th[2] = {sg, sg};
  double rel[2] = {1e300, 1e300}, best[2] = {1e300, 1e300};
  int stall[2] = {0, 0};
  for (int it = 0;; ++it) {
    // orthonormal basis
    {
      const double n1 = sqrt(block_norm2<NT>(x1, n, L.red));
      const double i1 = (n1 > 0.0) ? 1.0 / n1 : 1.0;
      zd d[1] = {czero<double>()};
      for (int r = red_first(); r < n; r += RT) {
        x1[r] = x1[r] * i1;
        d[0] = cfmac(d[0], x1[r], x2[r]);
      }
      block_reduce<NT, 1>(d, L.red);
      for (int r = t; r < n; r += NT) x2[r] = x2[r] - d[0] * x1[r];
      __syncthreads();
      const double n2 = sqrt(block_norm2<NT>(x2, n, L.red));
      const double i2 = (n2 > 0.0) ? 1.0 / n2 : 1.0;
      for (int r = t; r < n; r += NT) x2[r] = x2[r] * i2;
      __syncthreads();
    }
    pencil_apply<NT>(P, coef, ops, FORM_AM, sg, x1, a1, L.X1, L.X2, L.red);
    pencil_apply<NT>(P, coef, ops, FORM_BM, sg, x1, b1, L.X1, L.X2, L.red);
    pencil_apply<NT>(P, coef, ops, FORM_AM, sg, x2, a2, L.X1, L.X2, L.red);
    pencil_apply<NT>(P, coef, ops, FORM_BM, sg, x2, b2, L.X1, L.X2, L.red);
    // projected pencil: pa[i][j] = x_i^H a_j, pb[i][j] = x_i^H b_j
    zd pr[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) pr[k] = czero<double>();
    for (int r = red_first(); r < n; r += RT) {
      const zd u = x1[r], v = x2[r];
      pr[0] = cfmac(pr[0], u, a1[r]); pr[1] = cfmac(pr[1], u, a2[r]);
      pr[2] = cfmac(pr[2], v, a1[r]); pr[3] = cfmac(pr[3], v, a2[r]);
      pr[4] = cfmac(pr[4], u, b1[r]); pr[5] = cfmac(pr[5], u, b2[r]);
      pr[6] = cfmac(pr[6], v, b1[r]); pr[7] = cfmac(pr[7], v, b2[r]);
    }
    block_reduce<NT, 8>(pr, L.red);
    const zd A00 = pr[0], A01 = pr[1], A10 = pr[2], A11 = pr[3];
    const zd B00 = pr[4], B01 = pr[5], B10 = pr[6], B11 = pr[7];
    // det(A~ - theta B~) = qa theta^2 + qb theta + qc
    const zd qa = B00 * B11 - B01 * B10;
    const zd qb = czero<double>() - (A00 * B11 + A11 * B00 - A01 * B10 - A10 * B01);
    const zd qc = A00 * A11 - A01 * A10;
    if (!(cabs(qa) > 0.0)) break;            // B~ singular: leave rel at its last value
    {
      const zd sq = zsqrt(qb * qb - qa * qc * 4.0);
      // q = -(qb + s sq) / 2 with the sign that avoids cancellation
      const zd s1 = qb + sq, s2 = qb - sq;
      const zd q = (cabs(s1) >= cabs(s2) ? s1 : s2) * -0.5;
      const zd t0 = cdiv(q, qa), t1 = (cabs(q) > 0.0) ? cdiv(qc, q) : t0;
      // keep each pair's index from the previous step (its convergence state
      // is tracked per index)
      const bool swap = it > 0 && cabs(t0 - th[1]) + cabs(t1 - th[0]) < cabs(t0 - th[0]) + cabs(t1 - th[1]);
      th[0] = swap ? t1 : t0;
      th[1] = swap ? t0 : t1;
    }
    // 2-vectors y_k with (A~ - theta_k B~) y_k = 0, unit norm
    zd y[2][2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const zd m00 = A00 - th[k] * B00, m01 = A01 - th[k] * B01, m10 = A10 - th[k] * B10, m11 = A11 - th[k] * B11;
      zd y0 = czero<double>() - m01, y1 = m00;
      if (abs2(m11) + abs2(m10) > abs2(m00) + abs2(m01)) { y0 = m11; y1 = czero<double>() - m10; }
      double ny = sqrt(abs2(y0) + abs2(y1));
      if (!(ny > 0.0)) { y0 = mk(k == 0 ? 1.0 : 0.0, 0.0); y1 = mk(k == 0 ? 0.0 : 1.0, 0.0); ny = 1.0; }
      y[k][0] = y0 * (1.0 / ny);
      y[k][1] = y1 * (1.0 / ny);
    }
    // Ritz vectors into x1, x2 and residuals into a1, a2 (element-wise in place)
    zd nr[4] = {czero<double>(), czero<double>(), czero<double>(), czero<double>()};
    for (int r = red_first(); r < n; r += RT) {
      const zd u = x1[r], v = x2[r];
      const zd u0 = y[0][0] * u + y[0][1] * v, u1 = y[1][0] * u + y[1][1] * v;
      const zd r0 = (y[0][0] * a1[r] + y[0][1] * a2[r]) - th[0] * (y[0][0] * b1[r] + y[0][1] * b2[r]);
      const zd r1 = (y[1][0] * a1[r] + y[1][1] * a2[r]) - th[1] * (y[1][0] * b1[r] + y[1][1] * b2[r]);
      x1[r] = u0; x2[r] = u1; a1[r] = r0; a2[r] = r1;
      nr[0].x += abs2(u0); nr[1].x += abs2(u1); nr[2].x += abs2(r0); nr[3].x += abs2(r1);
    }
    block_reduce<NT, 4>(nr, L.red);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const double un = sqrt(nr[k].x), den = (nA + cabs(th[k]) * nB) * un;
      rel[k] = (den > 0.0) ? sqrt(nr[2 + k].x) / den : 1e300;
    }
    bool conv[2];
    double ffk[2] = {1.0, 1.0};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (rel[k] < 0.5 * best[k]) { best[k] = rel[k]; stall[k] = 0; } else if (rel[k] < 1e-12) { ++stall[k]; }
      conv[k] = rel[k] < tol || stall[k] >= 3;
    }
    // the farfield ratios enter only the choice of the wanted pair and the
    // early stop, which need a converged pair (conv comes from block-wide
    // sums, so the branch is the same for the whole work-group)
    if (conv[0] || conv[1]) {
#pragma unroll
      for (int k = 0; k < 2; ++k) ffk[k] = farfield_ratio<NT>(P, k == 0 ? x1 : x2, L.red);
    }
    int w;
    if (want == 1) {
      w = (cabs(th[0] - sg) <= cabs(th[1] - sg)) ? 0 : 1;
    } else {
      const bool d0 = lead2_discrete(P.alpha.x, th[0], ffk[0]), d1 = lead2_discrete(P.alpha.x, th[1], ffk[1]);
      w = (d0 && (!d1 || th[0].y >= th[1].y)) ? 0 : (d1 ? 1 : -1);
    }
    // early stop: the other pair is already an eigenpair to 1e-10 (so the
    // basis holds the two eigenvalues nearest the shift, not a passing mix)
    // and cannot outrank the converged wanted one
    bool done = conv[0] && conv[1];
    if (!done && w >= 0 && conv[w] && rel[w] < 1e-14 && rel[1 - w] < 1e-10) {
      const int o = 1 - w;
      done = !lead2_competes(want, P.alpha.x, sg, th[w], th[o], rel[o], ffk[o]);
    }
    if (done || it >= maxit) break;
    // corrections x_k = u_k - L(sigma)^-1 r_k: both solves in one pass over
    // the factors, in place in a1, a2 (scaled rows, zero padding)
    for (int r = t; r < P.npad; r += NT) {
      a1[r] = (r < n) ? a1[r] * dr[r] : czero<double>();
      a2[r] = (r < n) ? a2[r] * dr[r] : czero<double>();
    }
    __syncthreads();
    {
      zd *const ys[2] = {a1, a2};
      lu_solve_many<T, NT, 2, true>(P, A, ipiv, Lb, ys, tmp2, L.w2);
    }
    for (int r = t; r < n; r += NT) {
      x1[r] = x1[r] - a1[r] * dc[r];
      x2[r] = x2[r] - a2[r] * dc[r];
    }
    __syncthreads();
    nsolve += 2;
  }
  // ---- both Ritz vectors, getevec normalisation (first entry of largest
  // modulus set to 1), farfield ratio, out to columns 0 and 1
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    zd *x = (k == 0) ? x1 : x2;
    double bm = -1.0;
    int bi = 0x7fffffff;
    for (int r = t; r < n; r += NT) { const double a = abs2(x[r]); if (a > bm) { bm = a; bi = r; } }
    // all-NaN vector: no entry compares greater
    const zd scale = x[clamp_index(block_argmax<NT>(bm, bi, L.red), n)];
    __syncthreads();
    if (scale_ok(scale))
      for (int r = t; r < n; r += NT) x[r] = cdiv(x[r], scale);
    __syncthreads();
    const double ff = farfield_ratio<NT>(P, x, L.red);
    for (int r = t; r < n; r += NT) out[(size_t)k * nv + r] = x[r];
    if (t == 0) {
      eval2[2 * p + k] = th[k];
      resid2[2 * p + k] = rel[k];
      ff2[2 * p + k] = ff;
    }
  }
  if (t == 0) iters[p] += nsolve;
}


// ---------------------------------------------------------------------------
// Residual inverse iteration (A. Neumaier, "Residual inverse iteration for the
// nonlinear eigenvalue problem", SIAM J. Numer. Anal. 22 (1985) 914-923) for
// the eigenpair nearest the factored shift sigma:
//     x <- x - L(sigma)^-1 L(lambda) x,   lambda: root of x^H L(lambda) x = 0
// nearest the previous value, with L(l) = A - l B (temporal solver pencil) or
// C0 + l C1 + l^2 C2 (spatial, on phi directly).  The correction
// L(sigma)^-1 r shrinks with the residual r, so FP32 factors limit only the
// contraction per step (|lambda - sigma| / |lambda_2 - sigma| plus about
// kappa u32), not the attainable accuracy, which the FP64 residual sets.
// The first step is one plain inverse-iteration step x = L(sigma)^-1 L'(sigma) r
// from a hashed start vector.  One work-group per point.  Stops when the FP64
// relative residual is below tol, when it has not halved for three steps while
// below 1e-12 (the rounding floor), after maxit corrections, or (temporal
// points with a second pass to follow, from the sixth correction on, above
// 1e-12) when its rate over the last three steps predicts more than
// 3/4 (maxit + 1) solves in all.  Outputs per point: lambda, the
// vector normalised by its first entry of largest modulus (z = [phi;
// lambda phi] for spatial points, at out_off), the residual, the farfield
// ratio, the number of solves and a convergence flag (0, or 2 when the
// residual stayed above 1e-14).  pass2: 0 when no second pass follows, 1
// when k_invit2 follows, 2 when the work-group itself then runs the second
// pass (invit2_point) for a point that needs it (the launch then holds 2 NT
// more LDS entries).
// ---------------------------------------------------------------------------
template <typename T, int NB, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2))) void k_invit(const PointDev *__restrict__ pts, const cx<T> *__restrict__ mats,
                                              const int *__restrict__ pivs, const cx<T> *__restrict__ blks,
                                              const double *__restrict__ scales, const zd *__restrict__ coef,
                                              const double *__restrict__ ops, const double *__restrict__ norms,
                                              int maxit, double tol, zd *__restrict__ eval, zd *__restrict__ evec,
                                              double *__restrict__ resid, double *__restrict__ ffo,
                                              int *__restrict__ iters, int *__restrict__ flag, int npadmax,
                                              int nymax, const int *__restrict__ order, int pass2, int want,
                                              const int *__restrict__ info, zd *__restrict__ eval2,
                                              double *__restrict__ resid2, double *__restrict__ ff2) {
  extern __shared__ zd lds[];
  const int pi = order ? order[blockIdx.x] : blockIdx.x;   // largest points first
  const PointDev &P = pts[pi];
  OpLds L(lds, NT, npadmax, nymax, 1, npadmax);
  const int t = threadIdx.x, n = P.n;
  const cx<T> *A = mats + P.mat_off;
  const int *ipiv = pivs + P.piv_off;
  const cx<T> *Lb = blks + P.blk_off, *Ub = nullptr;
  const double *dr = scales + P.scale_off, *dc = dr + P.npad;
  const bool temporal = (P.itype == 1);
  const double nA = sqrt(norms[pi * 4 + 0]), nB = sqrt(norms[pi * 4 + 1]),
               nC = sqrt(norms[pi * 4 + 2]);
  const zd sg = P.shift;
  zd *x = L.z;

  // ---- start: x = L(sigma)^-1 L'(sigma) r
  const unsigned seed = point_seed(P);
  for (int r = t; r < n; r += NT) x[r] = mk(hash01(seed, 2 * r), hash01(seed, 2 * r + 1));
  __syncthreads();
  if (temporal) {
    pencil_apply<NT>(P, coef, ops, FORM_BM, sg, x, L.rhs, L.X1, L.X2, L.red);
  } else {
    pencil_apply<NT>(P, coef, ops, FORM_C1, sg, x, L.rhs, L.X1, L.X2, L.red);
    pencil_apply<NT>(P, coef, ops, FORM_C2, sg, x, L.res, L.X1, L.X2, L.red);
    for (int r = t; r < n; r += NT) L.rhs[r] = L.rhs[r] + (sg * 2.0) * L.res[r];
    __syncthreads();
  }
  shifted_solve<T, NB, NT, true>(P, A, ipiv, Lb, Ub, dr, dc, coef, ops, 0, L);
  for (int r = t; r < n; r += NT) x[r] = L.y[r];
  __syncthreads();
  int nsolve = 1;

  zd lam = sg;
  double rel = 1e300, best = 1e300;
  double back[3] = {1e300, 1e300, 1e300};   // rel one, two and three steps back
  int stall = 0;
  for (int it = 0;; ++it) {
    // unit 2-norm
    {
      const double nx = sqrt(block_norm2<NT>(x, n, L.red));
      const double inv = (nx > 0.0) ? 1.0 / nx : 1.0;
      for (int r = t; r < n; r += NT) x[r] = x[r] * inv;
      __syncthreads();
    }
    // pencil products and the new lambda
    zd d3[3] = {czero<double>(), czero<double>(), czero<double>()};
    if (temporal) {
      pencil_apply<NT>(P, coef, ops, FORM_AM, sg, x, L.y, L.X1, L.X2, L.red);
      pencil_apply<NT>(P, coef, ops, FORM_BM, sg, x, L.rhs, L.X1, L.X2, L.red);
      for (int r = red_first(); r < n; r += RT) {
        d3[0] = cfmac(d3[0], x[r], L.y[r]);
        d3[1] = cfmac(d3[1], x[r], L.rhs[r]);
      }
      block_reduce<NT, 3>(d3, L.red);
      if (cabs(d3[1]) > 0.0) lam = cdiv(d3[0], d3[1]);
    } else {
      pencil_apply<NT>(P, coef, ops, FORM_C0, sg, x, L.y, L.X1, L.X2, L.red);
      pencil_apply<NT>(P, coef, ops, FORM_C1, sg, x, L.rhs, L.X1, L.X2, L.red);
      pencil_apply<NT>(P, coef, ops, FORM_C2, sg, x, L.res, L.X1, L.X2, L.red);
      for (int r = red_first(); r < n; r += RT) {
        d3[0] = cfmac(d3[0], x[r], L.y[r]);
        d3[1] = cfmac(d3[1], x[r], L.rhs[r]);
        d3[2] = cfmac(d3[2], x[r], L.res[r]);
      }
      block_reduce<NT, 3>(d3, L.red);
      if (cabs(d3[2]) > 0.0) {
        const zd bb = cdiv(d3[1], d3[2] * 2.0), cc = cdiv(d3[0], d3[2]);
        const zd disc = bb * bb - cc;
        const double rr = cabs(disc);
        const double sr = sqrt(0.5 * (rr + fabs(disc.x)));
        zd sq;
        if (sr == 0.0) sq = czero<double>();
        else if (disc.x >= 0) sq = mk(sr, disc.y / (2.0 * sr));
        else sq = mk(fabs(disc.y) / (2.0 * sr), disc.y >= 0 ? sr : -sr);
        const zd r1 = czero<double>() - bb + sq, r2 = czero<double>() - bb - sq;
        lam = (cabs(r1 - lam) < cabs(r2 - lam)) ? r1 : r2;
      } else if (cabs(d3[1]) > 0.0) {
        lam = czero<double>() - cdiv(d3[0], d3[1]);
      }
    }
    // residual r = L(lambda) x into rhs
    zd part[1] = {czero<double>()};
    if (temporal) {
      for (int r = red_first(); r < n; r += RT) {
        const zd v = L.y[r] - lam * L.rhs[r];
        L.rhs[r] = v;
        part[0].x += abs2(v);
      }
    } else {
      const zd l2 = lam * lam;
      for (int r = red_first(); r < n; r += RT) {
        const zd v = L.y[r] + lam * L.rhs[r] + l2 * L.res[r];
        L.rhs[r] = v;
        part[0].x += abs2(v);
      }
    }
    block_reduce<NT, 1>(part, L.red);
    const double al = cabs(lam);
    const double den = temporal ? (nA + al * nB) : (nA + al * nB + al * al * nC);
    rel = sqrt(part[0].x) / den;             // ||x|| = 1
    // the stall count only runs near the rounding floor: far from it the
    // residual can grow for a step or two while the vector turns
    if (rel < 0.5 * best) { best = rel; stall = 0; } else if (rel < 1e-12) { ++stall; }
    // a temporal point that, at its rate over the last three steps, would
    // reach tol only after 3/4 of maxit + 1 solves (or not at all) leaves now
    // when a second pass follows: that pass takes such points whatever this
    // one gives them (a second eigenvalue nearly as close to the shift), so
    // the steps would be wasted
    bool slow = false;
    if (pass2 && temporal && it >= 6 && rel >= 1e-12 && rel >= tol) {
      const double rate = (back[2] > 0.0 && back[2] < 1e300) ? cbrt(rel / back[2]) : 1.0;
      slow = !(rate < 1.0) || nsolve + log(tol / rel) / log(rate) > 0.75 * (maxit + 1);
    }
    back[2] = back[1]; back[1] = back[0]; back[0] = rel;
    if (rel < tol || it >= maxit || stall >= 3 || slow) break;
    // correction
    shifted_solve<T, NB, NT, true>(P, A, ipiv, Lb, Ub, dr, dc, coef, ops, 0, L);
    ++nsolve;
    for (int r = t; r < n; r += NT) x[r] = x[r] - L.y[r];
    __syncthreads();
  }
  // ---- getevec normalisation: first entry of largest modulus set to 1
  double bm = -1.0;
  int bi = 0x7fffffff;
  for (int r = t; r < n; r += NT) { const double a = abs2(x[r]); if (a > bm) { bm = a; bi = r; } }
  // all-NaN vector: no entry compares greater
  const zd scale = x[clamp_index(block_argmax<NT>(bm, bi, L.red), n)];
  __syncthreads();
  if (scale_ok(scale))
    for (int r = t; r < n; r += NT) x[r] = cdiv(x[r], scale);
  __syncthreads();
  const double ff = farfield_ratio<NT>(P, x, L.red);
  zd *out = evec + P.out_off;
  for (int r = t; r < n; r += NT) {
    out[r] = x[r];
    if (!temporal) out[n + r] = lam * x[r];
  }
  if (t == 0) {
    eval[pi] = lam;
    resid[pi] = rel;
    ffo[pi] = ff;
    iters[pi] = nsolve;
    flag[pi] = (rel < 1e-14) ? 0 : 2;
  }
  // ---- the second pass in the same work-group (pass2 == 2), for the points the
  // rule of k_invit2 takes, with 2 maxit steps: it starts as soon as this
  // point's first pass ends, beside the other points' first passes.  x1 is
  // x (L.z), x2 L.res, a1 L.y, a2 L.rhs, b1 and b2 columns 2 and 3 of the
  // point's vector block, tmp2 the 2 NT entries after the operator layout.
  if (pass2 == 2 && lead2_needed(info[pi], P.itype, (rel < 1e-14) ? 0 : 2, want, P.alpha.x, lam, ff, nsolve, maxit)) {
    zd *tmp2 = NT > 256 ? L.tmp : lds + op_lds_bytes(npadmax, nymax, 1, npadmax) / sizeof(zd);
    const size_t nv = P.nvec;
    invit2_point<T, NB, NT>(P, pi, mats, pivs, blks, scales, coef, ops, norms, 2 * maxit, tol, want, eval2, evec,
                            resid2, ff2, iters, L, x, L.res, L.y, out + 2 * nv, L.rhs, out + 3 * nv, tmp2);
  }
}

// The second pass as a kernel of its own, after k_invit: one work-group per
// listed point p = sub[blockIdx.x], or per point order[blockIdx.x] that the
// rule takes.  LDS: the full operator layout followed by six npadmax vectors
// and 2 NT entries.
template <typename T, int NB, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2))) void k_invit2(const PointDev *__restrict__ pts, const int *__restrict__ sub,
                                               const cx<T> *__restrict__ mats, const int *__restrict__ pivs,
                                               const cx<T> *__restrict__ blks, const double *__restrict__ scales,
                                               const zd *__restrict__ coef, const double *__restrict__ ops,
                                               const double *__restrict__ norms, int maxit, double tol, int want,
                                               zd *__restrict__ eval2, zd *__restrict__ evec,
                                               double *__restrict__ resid2, double *__restrict__ ff2,
                                               int *__restrict__ iters, int npadmax, int nymax,
                                               const int *__restrict__ order, const int *__restrict__ info,
                                               const int *__restrict__ flag, const zd *__restrict__ eval1,
                                               const double *__restrict__ ff1, int maxit1) {
  extern __shared__ zd lds[];
  // sub lists the points; without it work-group g takes point order[g] and
  // runs only when the first pass (maxit1 steps) left that temporal point
  // unconverged, not discrete (unless want == 1), or converged only after
  // 3/4 of its steps -- the host applies the same rule to the same data
  const int p = sub ? sub[blockIdx.x] : order[blockIdx.x];
  if (!sub) {
    const PointDev &Q = pts[p];
    if (!lead2_needed(info[p], Q.itype, flag[p], want, Q.alpha.x, eval1[p], ff1[p], iters[p], maxit1)) return;
  }
  const PointDev &P = pts[p];
  OpLds L(lds, NT, npadmax, nymax, 1, npadmax);
  zd *x1 = L.X2 + 5 * nymax;
  zd *x2 = x1 + npadmax, *a1 = x2 + npadmax, *b1 = a1 + npadmax, *a2 = b1 + npadmax, *b2 = a2 + npadmax;
  zd *tmp2 = b2 + npadmax;                     // 2 NT entries for the two-column solve
  zd *out = evec + P.out_off;
  for (int r = threadIdx.x; r < P.n; r += NT) x1[r] = out[r];
  __syncthreads();
  invit2_point<T, NB, NT>(P, p, mats, pivs, blks, scales, coef, ops, norms, maxit, tol, want, eval2, evec, resid2,
                          ff2, iters, L, x1, x2, a1, b1, a2, b2, tmp2);
}

// Copy column sel[p] of each point's eigenvector block (P.out_off, nvec rows,
// ld nvec) to dst + doff[p].  grid: points; sel[p] < 0 skips the point.
__global__ __launch_bounds__(256) void k_gather_cols(const PointDev *__restrict__ pts, const zd *__restrict__ src,
                                                     const int *__restrict__ sel, const long long *__restrict__ doff,
                                                     zd *__restrict__ dst) {
  const PointDev &P = pts[blockIdx.x];
  const int k = sel[blockIdx.x];
  if (k < 0) return;
  const zd *s = src + P.out_off + (size_t)k * P.nvec;
  zd *d = dst + doff[blockIdx.x];
  for (int r = threadIdx.x; r < P.nvec; r += 256) d[r] = s[r];
}
