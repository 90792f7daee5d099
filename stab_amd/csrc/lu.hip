// Batched blocked complex LU with partial pivoting, one work-group per matrix
// (the getrf structure: factor a block column, swap, triangular solve, update).
//
// Columns are taken in blocks of KB = 64 (the last may be 32 wide).  Inside a
// block, panels of NB columns (16 in FP32, 8 in FP64) are factored with their rows in registers
// of the threads that own them (row r belongs to thread r % NT), so the pivot
// search and the rank-1 updates never touch memory.  Rows do not move while a
// block is factored: each thread tracks the position its rows would have
// after the interchanges so far (the pivot search compares positions, so the
// choice is the one of moved rows).  Each panel updates the rest of its block
// column in place, its rows of U being inv(L11) * A12.  When the block column
// is done its rows are put in their final order in one pass, and:
//   * its net row permutation is applied once to the trailing columns and,
//     for the LAPACK form only (left = 1), to the columns left of it;
//     otherwise it is stored as the block's interchange record for the solves,
//   * X = inv(L11) is formed once (four lanes per column, shuffles) and
//     stored as the block's inverse for the triangular solves, and U12 = X A12
//     runs on the matrix cores, and
//   * A22 -= L21 U12 with depth KB on the matrix cores, complex arithmetic as
//     2 x 2 real blocks, [Cr; Ci] -= [[Lr, -Li], [Li, Lr]] [Ur; Ui], i.e.
//     four real MFMA products per tile, computed transposed (the MFMA row index
//     runs over matrix columns) so that each accumulator register of 16 lanes
//     covers 16 consecutive matrix rows and loads/stores coalesce.
// The trailing matrix is read and written once per 64 columns.  P A = L U
// with P given by ipiv[].  Outputs: L and U in place, ipiv (absolute row
// indices, as ZGETRF), the pivot mode word and records (common.h), info and
// the inverses of the 64 x 64 diagonal blocks of L; k_blkinv then inverts
// those of U.  With left = 1 (pivot mode 0, the LAPACK form) L is in final
// row order and perm (ipiv + n, P as a row list) is stored too; with left = 0
// the columns left of each block keep their rows (mode 1).
#include "bounds.h"
#include "common.h"
#include <type_traits>
#include <utility>

// 16 x 16 x 4 MFMA: D[m][n] += sum_k A[m][k] B[k][n]; lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16].  Accumulator register i of lane l
// holds D[m][l % 16] with m = 4 (l / 16) + i (f32) or m = 4 i + l / 16 (f64).
template <typename T> struct Mfma;
template <> struct Mfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ inline v4 mac(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ inline int row_of(int lane, int i) { return 4 * i + (lane >> 4); }
  static constexpr int row_step(int i) { return 4 * i; }   // row_of(lane, i) - row_of(lane, 0)
};
template <> struct Mfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ inline v4 mac(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ inline int row_of(int lane, int i) { return 4 * (lane >> 4) + i; }
  static constexpr int row_step(int i) { return i; }       // row_of(lane, i) - row_of(lane, 0)
};

// Columns of one LDS tile of U12 in the MFMA update (f64: 32, f32: 64).
template <typename T> __host__ __device__ constexpr int lu_gw() { return sizeof(T) == 8 ? 32 : 64; }

// Elements of the diagonal-block inverse storage of one point (see k_blkinv).
__host__ __device__ inline long long blk_elems(int npad, int bs) {
  const long long nblk = (npad + bs - 1) / bs;
  return 2LL * nblk * bs * bs;
}

// f(0), ..., f(N - 1) with the index a compile-time constant in each
template <int... I, typename F> __device__ __forceinline__ void static_for_(std::integer_sequence<int, I...>, const F &f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(const F &f) {
  static_for_(std::make_integer_sequence<int, N>{}, f);
}

// Order the LDS accesses of one wave's lanes.
__device__ inline void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The wave's arg-max of (v, i): larger v, the lower i among equal v; v is a
// magnitude or -1 (no candidate).  The index comes back for the whole wave.
// Floats of these values order as their bits do, so the maximum is six integer
// DPP maxima of the (high) words; only where more than one lane holds it are
// the low words, then the indexes, compared.
__device__ inline int wave_max(int x) {
  constexpr int LOW = (int)0x80000000;
#define STAB_MAX_STEP(CTRL, RM) x = max(__builtin_amdgcn_update_dpp(LOW, x, CTRL, RM, 0xF, false), x);
  STAB_MAX_STEP(0x111, 0xF) STAB_MAX_STEP(0x112, 0xF) STAB_MAX_STEP(0x114, 0xF) STAB_MAX_STEP(0x118, 0xF)
  STAB_MAX_STEP(0x142, 0xA) STAB_MAX_STEP(0x143, 0xC)
#undef STAB_MAX_STEP
  return lane63(x);
}
__device__ inline int wave_best(int hi, unsigned lo, int i) {
  unsigned long long at = __ballot(hi == wave_max(hi));
  if (__builtin_expect((at & (at - 1)) != 0, 0)) {
    const int key = ((at >> (threadIdx.x & 63)) & 1ull) ? (int)(lo ^ 0x80000000u) : (int)0x80000000;
    at &= __ballot(key == wave_max(key));
    const int mi = ((at >> (threadIdx.x & 63)) & 1ull) ? ~i : (int)0x80000000;
    return ~wave_max(mi);
  }
  return __builtin_amdgcn_readlane(i, __builtin_ctzll(at));
}
__device__ inline int wave_best(float v, int i) { return wave_best(__float_as_int(v), 0u, i); }
__device__ inline int wave_best(double v, int i) {
  const long long b = __double_as_longlong(v);
  return wave_best((int)(b >> 32), (unsigned)b, i);
}

// 1 / b as cdiv(1, b) rounds it (zeros keep the signs that gives them), on one
// path: the larger component divides.
template <typename T> __device__ inline cx<T> crecip(cx<T> b) {
  const bool ge = fabs(b.x) >= fabs(b.y);
  const T big = ge ? b.x : b.y, sm = ge ? b.y : b.x;
  const T r = sm / big, d = fma(sm, r, big);
  const T nr = sizeof(T) == 4 ? -r : (T)0 - r;
  return mk<T>((ge ? (T)1 : r + (T)0) / d, (ge ? nr : (T)-1) / d);
}

// The batched LU in two launches per 64-column block (K0 = 0, 64, ...) over
// the whole batch:
//   k_lu_panel  one work-group per matrix whose order exceeds K0: factors the
//               block column [K0, K0 + kb) (panels in registers, the in-block
//               strips, on the matrix cores in FP32, the interchanges),
//               stores the block's records, and forms X = inv(L11); thread t
//               holds rows K0 + t + j NT, j < R, so R = ceil((n - K0) / NT)
//               suffices and later block steps launch with a smaller R;
//   k_lu_trail  one work-group per 64-column strip (32 in FP64) right of the
//               block, for every such matrix: the block's row permutation,
//               U12 = X A12 and A22 -= L21 U12 on the matrix cores.
// Split this way, the strips of one matrix run on several CUs at once and the
// latency-bound panel steps of some matrices overlap the matrix-core updates
// of others; the arithmetic is that of one work-group doing both in turn.
// A lone panel is bound by latency and by what one wave per SIMD issues: 64
// columns, each an arg-max, a publication through LDS, one barrier and a
// rank-1 update.  With rows that moved at every pivot, serial net permutations
// and strips of 16 columns loaded, updated and stored in turn, the panels of
// one matrix of order 480 took 1.65 ms in FP32 and 2.34 ms in FP64, now 0.82
// and 1.17 (256 such matrices: 1.88 and 2.92 ms, now 0.91 and 1.46).  While the
// accesses were flat ones (0.86 and 1.35 ms; see `at`) 0.38 and 0.41 ms were the
// columns, 0.17 and 0.55 A22, 0.11 and 0.12 X.  One row per thread fits the
// registers of three waves per SIMD; two rows would spill there, and ran 2-4%
// faster in those of two (800 matrices of order 480, flat accesses: 2.69 and
// 2.64 ms in FP32, 5.15 and 4.93 in FP64).
template <typename T, int NB, int NT, int R>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(R == 1 && NT == 256 ? 3 : 2))) void k_lu_panel(const PointDev *__restrict__ pts, cx<T> *__restrict__ mats,
                                                 int *__restrict__ pivs, cx<T> *__restrict__ blks,
                                                 int *__restrict__ info, const int *__restrict__ order, int left,
                                                 int K0) {
  typedef cx<T> C;
  // work-group -> point: `order` lists the points largest first, so the
  // batch's last work-groups are its cheapest
  const int pi = order[blockIdx.x];
  const PointDev &P = pts[pi];
  const int n = P.npad, lda = P.npad;
  if (K0 >= n) return;
  C *A = mats + P.mat_off;
  int *ipiv = pivs + P.piv_off;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  constexpr int NW = NT / 64;
  constexpr int KB = 64, SU = 2 * KB * 16, WS = KB - NB;    // WS: widest rest of the block column
  constexpr int NONE = 0x7fffffff;
  static_assert(KB % NB == 0, "panel width must divide the block width");
  static_assert(LU_PREC == 1 + 4 * KB, "interchange record: count, 2 KB rows, 2 KB sources");
  static_assert(LU_TREC == 1 + 3 * KB, "trailing record: count, KB top sources, KB out rows, KB out sources");

  // double-buffered by column parity: a column's slots are rewritten two
  // columns later, after a barrier every wave passes only once it has read
  // them.  Each wave publishes its best candidate and that row before the
  // column's one barrier.
  struct __attribute__((aligned(16))) Best { C inv; T v; int i; };   // a candidate: reciprocal, magnitude, position
  __shared__ C s_cand2[2][NW][NB];
  __shared__ Best s_best2[2][NW];
  __shared__ C s_blk[NB * NB];
  __shared__ C s_linv[NB * NB];           // inv(L11) of the current panel
  __shared__ int s_top[NB];               // rows (slots) of the panel's pivots
  __shared__ int s_srow[2 * KB], s_sorig[2 * KB];
  __shared__ int s_cnt[2][NW * R];
  __shared__ C s_u12[NB * WS];
  // staged A12 of the panel's pivot rows, then L21 in operand order (FP32);
  // packed strictly lower L11 for X (KB (KB - 1) / 2 entries); the left-column
  // interchanges (at most 2 KB rows x 16 columns); the final row list
  __shared__ C s_u[SU];
  static_assert(NB * WS <= SU, "A12 fits in s_u");

  C Pn[R][NB];
  int pos[R];                              // position of row K0 + t + j NT; NONE past the matrix
#pragma unroll
  for (int j = 0; j < R; ++j) pos[j] = (K0 + t + j * NT < n) ? K0 + t + j * NT : NONE;
  int mypiv = 0;                           // the pivot of column K0 + t
  int myinfo = (K0 == 0) ? 0 : info[pi];   // the first zero pivot of the earlier blocks

  const int kb = min(KB, n - K0);       // 64, or 32 for the last block (n is a multiple of 32)
  const int kend = K0 + kb;
  // row j of this thread (rows past the matrix: row K0), and its entry in a
  // column.  The column's address is uniform and passes through the asm so that
  // it stays a scalar of its own: 2 R NB whole addresses per lane, kept from the
  // loads to the stores, would spill.  The asm takes it as a global address: a
  // generic one comes back without its address space, and the accesses become
  // flat ones, which also count as LDS accesses where the wave waits.
  auto slot = [&](int j) { return K0 + t + j * NT < n ? K0 + t + j * NT : K0; };
  auto at = [&](int col, unsigned row) -> C & {
    typedef __attribute__((address_space(1))) char gchar;
    gchar *cp = (gchar *)(A + (size_t)col * lda);
    asm volatile("" : "+s"(cp));
    return *(C *)(cp + row * (unsigned)sizeof(C));
  };
  for (int k0 = K0; k0 < kend; k0 += NB) {
    // ---- load the panel (rows that were pivots earlier carry values that are
    // not used)
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int c = 0; c < NB; ++c) Pn[j][c] = at(k0 + c, slot(j));
    // ---- factor the panel; every register index is static, so the rank-1
    // updates touch only the columns right of the pivot
    static_for<NB>([&](auto cs) {
      constexpr int c = cs;
      const int col = k0 + c;
      T lv = (T)-1;
      int li = NONE;
      C lc = czero<T>();
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const T v = cabs1(Pn[j][c]);
        // a NaN never becomes a candidate; among equal magnitudes the lower position
        const bool up = (pos[j] >= col) & (pos[j] < NONE) & ((v > lv) | ((v == lv) & (pos[j] < li)));
        lv = up ? v : lv;
        li = up ? pos[j] : li;
        lc = mk<T>(up ? Pn[j][c].x : lc.x, up ? Pn[j][c].y : lc.y);
      }
      // every lane takes the reciprocal of its own candidate: a division is a
      // chain of dependent steps as the wave's arg-max is, and the two run
      // interleaved instead of one after the other
      const C rc = crecip(lc);
      const int bi = wave_best(lv, li);
      if (li == bi) {                       // the lane that holds the row at position bi (all, where none does)
        s_best2[c & 1][wv] = Best{rc, lv, li};
#pragma unroll
        for (int j = 0; j < R; ++j) {
          if (pos[j] == bi) {
#pragma unroll
            for (int cc = c + 1; cc < NB; ++cc) s_cand2[c & 1][wv][cc] = Pn[j][cc];
          }
        }
      }
      __syncthreads();
      Best b = s_best2[c & 1][0];
      int wb = 0;
#pragma unroll
      for (int w = 1; w < NW; ++w) {
        const Best o = s_best2[c & 1][w];
        const bool up = (o.v > b.v) | ((o.v == b.v) & (o.i < b.i));
        b.inv = mk<T>(up ? o.inv.x : b.inv.x, up ? o.inv.y : b.inv.y);
        b.v = up ? o.v : b.v;
        b.i = up ? o.i : b.i;
        wb = up ? w : wb;
      }
      if (__builtin_expect(__builtin_amdgcn_readfirstlane(b.i) == NONE, 0)) {
        // no candidate but NaN: keep the diagonal, whose reciprocal is NaN
        b.i = col;
        wb = 0;
        b.inv = mk<T>((T)__builtin_nan(""), (T)__builtin_nan(""));
        __syncthreads();
#pragma unroll
        for (int j = 0; j < R; ++j) {
          if (pos[j] == col) {
#pragma unroll
            for (int cc = c + 1; cc < NB; ++cc) s_cand2[c & 1][0][cc] = Pn[j][cc];
          }
        }
        __syncthreads();
      }
      const int p = b.i;
      mypiv = (t == col - K0) ? p : mypiv;
      const bool zero = b.v == (T)0;
      myinfo = (zero & (myinfo == 0)) ? col + 1 : myinfo;
      C u[NB];
#pragma unroll
      for (int cc = c + 1; cc < NB; ++cc) u[cc] = s_cand2[c & 1][wb][cc];
#pragma unroll
      for (int j = 0; j < R; ++j) {
        pos[j] = (pos[j] == p) ? col : (pos[j] == col ? p : pos[j]);
        if ((pos[j] > col) & (pos[j] < NONE) & !zero) {
          const C l = Pn[j][c] * b.inv;
          Pn[j][c] = l;
#pragma unroll
          for (int cc = c + 1; cc < NB; ++cc) Pn[j][cc] = cfms(Pn[j][cc], l, u[cc]);
        }
      }
    });
    // ---- write the factored panel back (rows still in place); stage the
    // diagonal block
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if (pos[j] >= k0 && pos[j] < NONE) {
#pragma unroll
        for (int c = 0; c < NB; ++c) at(k0 + c, slot(j)) = Pn[j][c];
        if (pos[j] < k0 + NB) {
          s_top[pos[j] - k0] = slot(j);
#pragma unroll
          for (int c = 0; c < NB; ++c) s_blk[(pos[j] - k0) * NB + c] = Pn[j][c];
        }
      }
    }
    __syncthreads();
    const int c0 = k0 + NB, w = kend - c0;      // the rest of the block column
    if (w <= 0) break;
    // ---- A12: the pivot rows of the rest, staged by the waves after the
    // first, while the first forms inv(L11) (unit lower): four lanes per column
    // c, lane q of them with the rows i = q (mod 4) in registers, term k of every
    // row as soon as x[k] is known (the terms k < c vanish: x[k] = 0 there).  With
    // a lane per column the panels took 1.12 and 1.90 ms (256 of order 480).
    if (wv == 0) {
      if (lane < 4 * NB) {
        const int c = lane >> 2, q = lane & 3;
        C x[NB / 4];
#pragma unroll
        for (int m = 0; m < NB / 4; ++m) x[m] = mk<T>((T)(4 * m + q == c), 0);
        static_for<NB - 1>([&](auto ks) {
          constexpr int k = ks, mk_ = k / 4, qk = k % 4;
          C xk = mk<T>(dpp_move<0x55 * qk>(x[mk_].x), dpp_move<0x55 * qk>(x[mk_].y));
          xk = mk<T>(k < c ? (T)0 : xk.x, k < c ? (T)0 : xk.y);
#pragma unroll
          for (int m = mk_; m < NB / 4; ++m) {
            const C l = s_blk[(4 * m + q) * NB + k];
            const C v = cfms(x[m], mk<T>(k < c ? (T)0 : l.x, k < c ? (T)0 : l.y), xk);
            const bool up = m > mk_ || q > qk;          // rows below k only
            x[m] = mk<T>(up ? v.x : x[m].x, up ? v.y : x[m].y);
          }
        });
#pragma unroll
        for (int m = 0; m < NB / 4; ++m) {
          const int i = 4 * m + q;
          s_linv[i * NB + c] = mk<T>(i < c ? (T)0 : x[m].x, i < c ? (T)0 : x[m].y);
        }
      }
    } else {
      for (int e = t - 64; e < NB * w; e += NT - 64) {
        const int i = e % NB, cc = e / NB;
        s_u[i * WS + cc] = A[(size_t)(c0 + cc) * lda + s_top[i]];
      }
    }
    __syncthreads();
    for (int e = t; e < NB * w; e += NT) {
      const int cc = e / NB, i = e - cc * NB;     // consecutive lanes: rows of one column
      C u = czero<T>();
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const C v = s_u[k * WS + cc];
        if (k <= i) u = cfma(u, s_linv[i * NB + k], v);
      }
      s_u12[i * WS + cc] = u;
      A[(size_t)(c0 + cc) * lda + s_top[i]] = u;
    }
    __syncthreads();
    // ---- A22 -= L21 U12 on the rows below the panel, wherever they are.
    if constexpr (sizeof(T) == 4 && NB == 16 && 32 * NB * NW <= SU) {
      // FP32, on the matrix cores, as the trailing kernel does it (C tile = the
      // update transposed: lane l holds columns 4 (l / 16) + i of row r0 + l % 16).
      // The B operand L21(r0 + l % 16, 4 s + l / 16) belongs to another lane of
      // the wave, so each wave stages the L21 rows of two tiles (32 rows x NB)
      // in its part of s_u and reads them back in operand order; the column
      // tiles of a row tile are loaded together.  Rows at or above the panel
      // are computed with the others and not stored.
      typedef typename Mfma<T>::v4 v4;
      C *lst = s_u + (size_t)wv * 32 * NB;
      const int nct = w / 16;
      static_for<R>([&](auto js) {
        constexpr int j = js;
        const int w0 = K0 + 64 * wv + j * NT;
        const unsigned long long live = __ballot(pos[j] >= c0 && pos[j] < NONE);
#pragma unroll 1
        for (int half = 0; half < 2; ++half) {
          const unsigned lm = (unsigned)(live >> (32 * half));
          if (lm == 0) continue;                                   // wave-uniform
          wave_lds_order();
          if ((lane >> 5) == half) {
#pragma unroll
            for (int k = 0; k < NB; ++k) lst[(lane & 31) * NB + k] = Pn[j][k];
          }
          wave_lds_order();
#pragma unroll 1
          for (int a = 0; a < 2; ++a) {
            const unsigned am = (lm >> (16 * a)) & 0xffffu;
            if (am == 0) continue;                                 // wave-uniform
            const bool st_ok = (am >> (lane & 15)) & 1u;
            const int r0 = w0 + 32 * half + 16 * a;
            C *Ab = A + (size_t)(c0 + 4 * (lane >> 4)) * lda + r0 + (lane & 15);
            v4 dr[WS / 16], di[WS / 16];
#pragma unroll
            for (int ct = 0; ct < WS / 16; ++ct)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const C x = Ab[(size_t)(min(ct, nct - 1) * 16 + i) * lda];
                dr[ct][i] = x.x;
                di[ct][i] = x.y;
              }
            C l[NB / 4];
#pragma unroll
            for (int st = 0; st < NB / 4; ++st) l[st] = lst[(16 * a + (lane & 15)) * NB + 4 * st + (lane >> 4)];
#pragma unroll
            for (int ct = 0; ct < WS / 16; ++ct) {
              if (ct >= nct) break;
#pragma unroll
              for (int st = 0; st < NB / 4; ++st) {
                const C u = s_u12[(4 * st + (lane >> 4)) * WS + ct * 16 + (lane & 15)];
                const T nur = -u.x, ui = u.y, nui = -u.y;
                dr[ct] = Mfma<T>::mac(nur, l[st].x, dr[ct]);
                dr[ct] = Mfma<T>::mac(ui, l[st].y, dr[ct]);
                di[ct] = Mfma<T>::mac(nui, l[st].x, di[ct]);
                di[ct] = Mfma<T>::mac(nur, l[st].y, di[ct]);
              }
              if (st_ok) {
#pragma unroll
                for (int i = 0; i < 4; ++i) Ab[(size_t)(ct * 16 + i) * lda] = mk<T>(dr[ct][i], di[ct][i]);
              }
            }
          }
        }
      });
    } else {
      // FP64 (and 512 threads, whose staging would not fit in s_u), on the VALU
      // (the FP64 matrix cores gave the same sums, 1.42 ms against 1.37 on flat
      // accesses): G columns of a row at a time, the next group's entries loaded
      // while one is computed
      constexpr int G = 4;
      static_for<R>([&](auto js) {
        constexpr int j = js;
        if (__ballot(pos[j] >= c0 && pos[j] < NONE) == 0) return;
        const bool live = pos[j] >= c0 && pos[j] < NONE;
        C nx[G];
#pragma unroll
        for (int q = 0; q < G; ++q) nx[q] = at(c0 + q, slot(j));
#pragma unroll 1
        for (int cg = 0; cg < w; cg += G) {
          C acc[G];
#pragma unroll
          for (int q = 0; q < G; ++q) acc[q] = nx[q];
#pragma unroll
          for (int q = 0; q < G; ++q) nx[q] = at(c0 + min(cg + G, w - G) + q, slot(j));
#pragma unroll
          for (int k = 0; k < NB; ++k)
#pragma unroll
            for (int q = 0; q < G; ++q) acc[q] = cfms(acc[q], Pn[j][k], s_u12[k * WS + cg + q]);
          if (live) {
#pragma unroll
            for (int q = 0; q < G; ++q) at(c0 + cg + q, slot(j)) = acc[q];
          }
        }
      });
    }
    __syncthreads();
  }  // panels of the block

  // ---- the interchanges: ipiv, and the block's net permutation (position
  // pos[j] receives row slot(j)) as the record of the forward solves (every row
  // that moves; read in pivot mode 1) and the trailing record of the update
  // kernel (the input row of each block-top row, the rows below that change).
  // List places in row order: counts per (j, wave), then ballot ranks.
  if (t < kb) ipiv[K0 + t] = mypiv;
  unsigned long long mm[R], mo[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const bool moved = pos[j] < NONE && pos[j] != slot(j);
    mm[j] = __ballot(moved);
    mo[j] = __ballot(moved && pos[j] >= kend);
    if (lane == 0) {
      s_cnt[0][j * NW + wv] = __builtin_popcountll(mm[j]);
      s_cnt[1][j * NW + wv] = __builtin_popcountll(mo[j]);
    }
  }
  __syncthreads();
  int bns = 0, bnout = 0;
  {
    int *rec = ipiv + 2 * n + 1 + (size_t)(K0 / KB) * LU_PREC;
    int *trec = ipiv + lu_trec_off(n, K0 / KB);
    const unsigned long long before = (1ull << lane) - 1ull;
    static_for<R>([&](auto js) {
      constexpr int j = js;
      int e = bns, o = bnout;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const int cm = s_cnt[0][j * NW + w], co = s_cnt[1][j * NW + w];
        e += w < wv ? cm : 0;
        o += w < wv ? co : 0;
        bns += cm;
        bnout += co;
      }
      const int row = slot(j);
      if (pos[j] < kend) trec[1 + pos[j] - K0] = row;
      if ((mm[j] >> lane) & 1ull) {
        e += __builtin_popcountll(mm[j] & before);
        s_srow[e] = pos[j];
        s_sorig[e] = row;
        rec[1 + e] = pos[j];
        rec[1 + 2 * KB + e] = row;
        if (pos[j] >= kend) {
          o += __builtin_popcountll(mo[j] & before);
          trec[1 + KB + o] = pos[j];
          trec[1 + 2 * KB + o] = row;
        }
      }
    });
    if (t == 0) { rec[0] = bns; trec[0] = bnout; }
  }
  // ---- the block's rows into their final order, MC columns at a time: every
  // moving row is read before any is written
  constexpr int MC = 8;
  for (int c0 = K0; c0 < kend; c0 += MC) {
    T vx[R][MC], vy[R][MC];
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int c = 0; c < MC; ++c) {
        const C v = at(c0 + c, slot(j));
        vx[j][c] = v.x;
        vy[j][c] = v.y;
      }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < R; ++j)
      if ((mm[j] >> lane) & 1ull) {
#pragma unroll
        for (int c = 0; c < MC; ++c) at(c0 + c, pos[j]) = mk<T>(vx[j][c], vy[j][c]);
      }
  }
  __syncthreads();
  // ---- left columns [0, K0) (pivot mode 0 only): move the touched rows,
  // 16 columns at a time, through LDS (bns * 16 <= 2 KB * 16 = SU entries)
  if (left && bns > 0 && K0 > 0) {
    for (int c0 = 0; c0 < K0; c0 += 16) {
      for (int e = t; e < bns * 16; e += NT) s_u[e] = A[(size_t)(c0 + e / bns) * lda + s_sorig[e % bns]];
      __syncthreads();
      for (int e = t; e < bns * 16; e += NT) A[(size_t)(c0 + e / bns) * lda + s_srow[e % bns]] = s_u[e];
      __syncthreads();
    }
  }
  // ---- X = inv(L11) (unit lower, zero outside kb x kb) in T arithmetic,
  // column-major into this block's slot of the diagonal-block inverses
  // (read by the triangular solves, and below by U12 = X A12).  Four lanes
  // per column: lane q of column c keeps x[m] = X(4 m + q, c) in registers
  // and sums the terms k = q (mod 4) of each substitution step; the sums meet
  // by shuffles.  The strictly lower triangle of L11 is staged in s_u, packed
  // by rows (row i at i (i - 1) / 2; 2016 entries), with zeros in rows and
  // columns past kb.
  C *X = blks + P.blk_off + (size_t)(K0 / KB) * KB * KB;
  static_assert(KB * (KB - 1) / 2 <= SU, "packed L11 fits in s_u");
  for (int e = t; e < KB * KB; e += NT) {
    const int i = e % KB, k = e / KB;
    if (k < i) {
      const C v = A[lu_l11_src(K0, kb, i, k, lda)];
      s_u[i * (i - 1) / 2 + k] = (i < kb) ? v : czero<T>();
    }
  }
  __syncthreads();
  if (t < 4 * KB) {
    const int c = t >> 2, q = t & 3;
    C x[KB / 4];
#pragma unroll
    for (int m = 0; m < KB / 4; ++m) x[m] = czero<T>();
#pragma unroll
    for (int mi = 0; mi < KB / 4; ++mi) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * mi + r;
        C s = czero<T>();
#pragma unroll
        for (int m = 0; m <= mi; ++m)     // entry (i, 4 m + q) of L11 when 4 m + q < i
          s = cfma(s, (m < mi || q < r) ? s_u[i * (i - 1) / 2 + 4 * m + q] : czero<T>(), x[m]);
        s.x += quad_xor1(s.x); s.y += quad_xor1(s.y);
        s.x += quad_xor2(s.x); s.y += quad_xor2(s.y);
        const C v = (i < c || i >= kb || c >= kb) ? czero<T>() : ((i == c) ? mk<T>(1, 0) : czero<T>() - s);
        if (r == q) x[mi] = v;
      }
    }
#pragma unroll
    for (int m = 0; m < KB / 4; ++m) X[c * KB + 4 * m + q] = x[m];
  }
  __syncthreads();
  // ---- final row permutation: row r of L U is row perm[r] of the input,
  // composed in LDS by one thread, then stored; only the LAPACK form (pivot
  // mode 0) has it: the mode-1 solves use the block records
  static_assert(sizeof(s_u) >= 2 * 1280 * sizeof(int), "two row lists fit in s_u");
  if (left && kend == n) {
    int *perm = ipiv + n;
    int *s_ip = reinterpret_cast<int *>(s_u), *s_slot = s_ip + 1280;   // the pivots, the rows
    __syncthreads();
    for (int r = t; r < n; r += NT) { s_slot[r] = r; s_ip[r] = ipiv[r]; }
    __syncthreads();
    if (t == 0) {
      for (int c = 0; c < n; ++c) {
        const int p = s_ip[c];
        if (p != c) { const int a = s_slot[c]; s_slot[c] = s_slot[p]; s_slot[p] = a; }
      }
    }
    __syncthreads();
    for (int r = t; r < n; r += NT) perm[r] = s_slot[r];
  }
  if (t == 0) {
    info[pi] = myinfo;
    if (kend == n) ipiv[2 * n] = left ? 0 : 1;
  }
}


// Strip [c0, c0 + gw) of the columns right of block K0 of one matrix
// (tasks[2 b], tasks[2 b + 1] = point, c0; point -1 pads the grid): stage the
// block rows of the strip in final order (some come from below the block;
// the rows below that change then receive their input rows, which lie in
// the block top and are not written before U12 is stored), U12 = X S with
// X = inv(L11) of the block, and A22 -= L21 U12 over the rows below the
// block.  Complex products as 2 x 2 real blocks on the matrix cores,
// computed transposed (MFMA rows = matrix columns) so that each accumulator
// register of 16 lanes covers 16 consecutive matrix rows.
// Streaming load of one A22 entry: the trailing update reads each A22 tile
// once per block step and writes it back with store_stream (the next read is
// a block step later, after the batch's other tiles have passed through the
// caches), so L2 is left to the L21 panel that every strip of a point reads.
template <typename T> __device__ inline cx<T> load_stream(const cx<T> *p);
template <> __device__ inline zf load_stream<float>(const zf *p) {
  typedef float v2 __attribute__((ext_vector_type(2)));
  const v2 w = __builtin_nontemporal_load((const v2 *)p);
  return mk(w.x, w.y);
}
template <> __device__ inline zd load_stream<double>(const zd *p) {
  typedef double v2 __attribute__((ext_vector_type(2)));
  const v2 w = __builtin_nontemporal_load((const v2 *)p);
  return mk(w.x, w.y);
}
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_lu_trail(const PointDev *__restrict__ pts, cx<T> *__restrict__ mats,
                                                  const int *__restrict__ pivs, const cx<T> *__restrict__ blks,
                                                  const int *__restrict__ tasks, int K0) {
  typedef cx<T> C;
  typedef typename Mfma<T>::v4 v4;
  constexpr int NT = 256, NW = NT / 64, KB = 64, GW = lu_gw<T>(), UP = GW + 1, CT = GW / 16;
  const int pi = tasks[2 * blockIdx.x], c0 = tasks[2 * blockIdx.x + 1];
  if (pi < 0) return;
  const PointDev &P = pts[pi];
  const int n = P.npad, lda = P.npad;
  if (K0 >= n) return;
  const int kb = min(KB, n - K0), kend = K0 + kb;
  if (c0 < kend || c0 >= n) return;
  C *A = mats + P.mat_off;
  const int *trec = pivs + P.piv_off + lu_trec_off(n, K0 / KB);
  const C *X = blks + P.blk_off + (size_t)(K0 / KB) * KB * KB;
  // the wave index as a scalar: the row offsets of the update below are then
  // wave-uniform and the addresses a per-lane base plus a scalar offset
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
  __shared__ int s_topsrc[KB], s_outrow[KB], s_outsrc[KB];
  __shared__ C s_u[KB * UP];
  const int nout = min(trec[0], KB);
  for (int e = t; e < kb; e += NT) s_topsrc[e] = trec[1 + e];
  for (int e = t; e < nout; e += NT) { s_outrow[e] = trec[1 + KB + e]; s_outsrc[e] = trec[1 + 2 * KB + e]; }
  __syncthreads();
  const int gw = min(GW, n - c0);
  // stage the block rows of the strip in final order (some come from
  // below the block); then the rows below that change receive their
  // input rows, which lie in the block top and are not written before
  // U12 is stored
  {
    // every load of the thread issued before the first store to LDS
    constexpr int NE = (KB * GW + NT - 1) / NT;
    C v[NE];
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const int e = t + q * NT, k = e % KB, j = e / KB;
      const bool ok = k < kb && j < gw;       // else a harmless in-range load, not stored
      v[q] = A[(size_t)(ok ? c0 + j : c0) * lda + (ok ? s_topsrc[k] : K0)];
    }
#pragma unroll
    for (int q = 0; q < NE; ++q) {
      const int e = t + q * NT, k = e % KB, j = e / KB;
      if (k < kb && j < gw) s_u[k * UP + j] = v[q];
    }
  }
  __syncthreads();
  for (int e = t; e < nout * gw; e += NT) {
    const int o = e % nout, j = e / nout;
    A[(size_t)(c0 + j) * lda + s_outrow[o]] = A[(size_t)(c0 + j) * lda + s_outsrc[o]];
  }
  // U12 = X S (S = the staged rows) on the matrix cores, transposed as
  // the update below: wave w takes column tile w % CTN and the row tiles
  // it owns (four per column tile, split over NW / CTN waves so that the
  // triangular work, 4 (rt + 1) depth-4 steps for row tile rt, balances)
  {
    constexpr int CTN = GW / 16, NWC = NW / CTN;
    static_assert(NWC == 1 || NWC == 2 || NWC == 4, "waves per U12 column tile");
    const C *Xs = X;
    const int ct = wv % CTN, h = wv / CTN;
    const bool colok = ct * 16 < gw;
    v4 ur[4], ui[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) { ur[rt][i] = (T)0; ui[rt][i] = (T)0; }
      const int own = (NWC == 1) ? 0 : (NWC == 2 ? ((rt == 0 || rt == 3) ? 0 : 1) : rt);
      if (own != h || !colok) continue;
      // X(i, k) = 0 for k > i: row tile rt needs k < 16 (rt + 1)
#pragma unroll
      for (int ks = 0; ks < 4 * (rt + 1); ++ks) {
        const int k = 4 * ks + (lane >> 4);
        const C sv = s_u[k * UP + ct * 16 + (lane & 15)];
        const C xv = Xs[(size_t)k * KB + rt * 16 + (lane & 15)];
        ur[rt] = Mfma<T>::mac(sv.x, xv.x, ur[rt]);
        ur[rt] = Mfma<T>::mac(-sv.y, xv.y, ur[rt]);
        ui[rt] = Mfma<T>::mac(sv.y, xv.x, ui[rt]);
        ui[rt] = Mfma<T>::mac(sv.x, xv.y, ui[rt]);
      }
    }
    __syncthreads();     // S fully read
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const int own = (NWC == 1) ? 0 : (NWC == 2 ? ((rt == 0 || rt == 3) ? 0 : 1) : rt);
      if (own != h || !colok) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = ct * 16 + Mfma<T>::row_of(lane, i), row = rt * 16 + (lane & 15);
        if (j < gw) {
          const C u = mk<T>(ur[rt][i], ui[rt][i]);
          s_u[row * UP + j] = u;
          A[(size_t)(c0 + j) * lda + K0 + row] = u;
        }
      }
    }
    __syncthreads();
  }
  // A22 -= L21 U12: each wave takes chunks of 16 rows against the gw columns
  // of the strip (rows of all chunks are multiples of 16 below n, a multiple
  // of 32); the A22 tile of the wave's next chunk is loaded while the current
  // one is on the matrix cores
  // Addresses as one per-lane base plus wave-uniform offsets: tile entry
  // (ct, i) of rows r0 .. r0 + 15 is Ab[(ct 16 + row_step(i)) lda + r0], and
  // L21 entry of depth step s is Lb[(4 s) lda + r0].  Loads take clamped
  // in-range offsets and are selected afterwards, so none waits under a branch.
  const C *Lb = A + (size_t)(K0 + (lane >> 4)) * lda + (lane & 15);
  C *Ab = A + (size_t)(c0 + Mfma<T>::row_of(lane, 0)) * lda + (lane & 15);
  v4 dr[CT], di[CT], nr[CT], ni[CT];
  int r0 = kend + 16 * wv;
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool ok = r0 < n && ct * 16 < gw;
      C x = load_stream(Ab + (ok ? (ct * 16 + Mfma<T>::row_step(i)) * lda + r0 : kend));
      if (!ok) x = czero<T>();
      dr[ct][i] = x.x;
      di[ct][i] = x.y;
    }
  for (; r0 < n; r0 += 16 * NW) {
    const int rn = r0 + 16 * NW;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool ok = rn < n && ct * 16 < gw;
        C x = load_stream(Ab + (ok ? (ct * 16 + Mfma<T>::row_step(i)) * lda + rn : r0));
        if (!ok) x = czero<T>();
        nr[ct][i] = x.x;
        ni[ct][i] = x.y;
      }
    // L21 of the chunk is loaded LH depth-4 steps at a time before the
    // MFMA chain that uses it (one memory latency per LH steps).  kb is 32 or
    // 64, so every step of a 4 LH = 32 deep pass is inside the block; the
    // column tiles past gw (the last strip of an order 32 mod 64) are
    // computed from in-range data and not stored: a guard here would split
    // the MFMA chain into branches that copy its accumulators
    constexpr int LH = 8;
    static_assert(4 * LH == 32, "kb is a multiple of 32");
#pragma unroll 1
    for (int kb0 = 0; kb0 < kb; kb0 += 4 * LH) {
      T lr[LH], li[LH];
#pragma unroll
      for (int st = 0; st < LH; ++st) {
        const C x = Lb[(kb0 + 4 * st) * lda + r0];
        lr[st] = x.x;
        li[st] = x.y;
      }
#pragma unroll
      for (int st = 0; st < LH; ++st) {
        const int k = kb0 + 4 * st + (lane >> 4);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const C uu = s_u[k * UP + ct * 16 + (lane & 15)];
          const T nur = -uu.x, ui = uu.y, nui = -uu.y;
          dr[ct] = Mfma<T>::mac(nur, lr[st], dr[ct]);
          dr[ct] = Mfma<T>::mac(ui, li[st], dr[ct]);
          di[ct] = Mfma<T>::mac(nui, lr[st], di[ct]);
          di[ct] = Mfma<T>::mac(nur, li[st], di[ct]);
        }
      }
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (ct * 16 < gw) store_stream(Ab + (ct * 16 + Mfma<T>::row_step(i)) * lda + r0, mk<T>(dr[ct][i], di[ct][i]));
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) { dr[ct] = nr[ct]; di[ct] = ni[ct]; }
  }
}

// Inverses of the diagonal blocks of U (upper) of order BS = 64 (the last
// block may be shorter; entries outside it are stored as zeros), in FP64
// arithmetic, stored as T, column-major.  With nblk = ceil(npad / BS), block b
// of inv(L) is at blk_off + b BS^2 (written by k_lu_panel) and block b
// of inv(U) at blk_off + (nblk + b) BS^2; the per-point allocation is
// 2 nblk BS^2 elements (blk_elems above).
// grid: x = block index, y = point; 256 threads, four lanes per column: lane
// q of column c sums the terms k = q (mod 4) of each substitution step and
// keeps the entries x[k][c], k = q (mod 4), in registers; the step's sum is
// reduced over the four lanes by shuffles, so the 64-step recurrence needs
// no barrier.  The reciprocals of the 64 diagonal entries are formed once,
// in LDS, so each step multiplies instead of dividing.  Besides them only the
// block itself lives in LDS, as stored (the arithmetic converts to FP64).
template <typename T, int BS>
__global__ __launch_bounds__(4 * BS) void k_blkinv(const PointDev *__restrict__ pts, const cx<T> *__restrict__ mats,
                                                   cx<T> *__restrict__ blks) {
  static_assert(BS == 64, "four lanes per column of a 64-wide block");
  const PointDev &P = pts[blockIdx.y];
  const int n = P.npad, k0 = blockIdx.x * BS;
  if (k0 >= n) return;
  const int bs = min(BS, n - k0), t = threadIdx.x;
  const int nblk = (n + BS - 1) / BS;
  const cx<T> *A = mats + P.mat_off;
  cx<T> *Ui = blks + P.blk_off + (size_t)(nblk + blockIdx.x) * BS * BS;
  constexpr int LD = BS + 1;       // padded rows: the column-wise staging writes hit distinct banks
  __shared__ cx<T> s_a[BS * LD];  // row-major copy of the block, as stored (FP32: 33 KB, so more groups per CU)
  __shared__ zd s_rd[BS];          // 1 / U(i, i)
  for (int e = t; e < BS * BS; e += 4 * BS) {
    const int i = e % BS, j = e / BS;   // consecutive lanes read consecutive rows of column j
    const bool ok = i < bs && j < bs;
    const cx<T> v = A[(size_t)(k0 + (ok ? j : 0)) * n + k0 + (ok ? i : 0)];
    s_a[i * LD + j] = ok ? v : czero<T>();
  }
  if (t < BS) {
    const int i = min(t, bs - 1);
    s_rd[t] = cdiv(mk(1.0, 0.0), cvt<double>(A[(size_t)(k0 + i) * n + k0 + i]));
  }
  __syncthreads();
  const int c = t >> 2, q = t & 3;
  zd x[BS / 4];                   // x[m] = entry (4 m + q, c) of the inverse being built
  // inv(U) column c: x_i = (delta_ic - sum_{i < k <= c} U_ik x_k) / U_ii, i = c .. 0
#pragma unroll
  for (int m = 0; m < BS / 4; ++m) x[m] = czero<double>();
#pragma unroll
  for (int mi = BS / 4 - 1; mi >= 0; --mi) {
#pragma unroll
    for (int r = 3; r >= 0; --r) {
      const int i = 4 * mi + r;
      zd s = czero<double>();
#pragma unroll
      for (int m = mi; m < BS / 4; ++m) {
        const int k = 4 * m + q;
        if (k > i && k <= c) s = cfma(s, cvt<double>(s_a[i * LD + k]), x[m]);
      }
      s.x += quad_xor1(s.x); s.y += quad_xor1(s.y);
      s.x += quad_xor2(s.x); s.y += quad_xor2(s.y);
      const zd rhs = ((i == c) ? mk(1.0, 0.0) : czero<double>()) - s;
      const zd v = (i > c || c >= bs) ? czero<double>() : rhs * s_rd[i];
      if (r == q) x[mi] = v;
    }
  }
#pragma unroll
  for (int m = 0; m < BS / 4; ++m) Ui[c * BS + 4 * m + q] = cvt<T>(x[m]);
}
