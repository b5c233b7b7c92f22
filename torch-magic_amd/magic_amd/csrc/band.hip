// Pivoted band LU in LINPACK dgbfa/dgbsl order for the finite-difference
// per-degree systems.  Band storage abd[(2kl+ku+1) x n] (row kl+ku is the
// diagonal, the first kl rows hold fill-in), multipliers stored negated,
// pivots 1-based, singular pivot threshold 1e-15.  The factorisation is
// sequential in the column index by nature: one wave factors one matrix held
// in LDS (one lane per matrix when the band does not fit in 64 KB).  The solve
// runs all right-hand-side rows of all degrees in one launch, each row using
// its degree's factors, over coalesced LDS tiles.  Band widths up to kl, ku = 4
// (the 9-band double-curl operator) are supported by the solve.
#include "common.h"

#include <type_traits>

#define AB(i, j) abd[(long)(i) * n + (j)]  // 0-based band row i, column j

__global__ void k_band_factor(double* __restrict__ abd_all, int* __restrict__ piv_all,
                              int* __restrict__ info_all, int n, int kl, int ku, int nbatch,
                              const int* when) {
  if (when && *when == 0) return;
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbatch) return;
  const int nrow = 2 * kl + ku + 1;
  double* abd = abd_all + (long)b * nrow * n;
  int* pivot = piv_all + (long)b * n;
  const int m = kl + ku + 1;  // 1-based diagonal row
  int info = 0;
  const int j0 = ku + 2, j1 = (n < m ? n : m) - 1;
  for (int jz = j0; jz <= j1; ++jz)
    for (int i = m + 1 - jz; i <= kl; ++i) AB(i - 1, jz - 1) = 0.0;
  int jz = j1, ju = 0;
  for (int k = 1; k <= n - 1; ++k) {
    const int kp1 = k + 1;
    jz = jz + 1;
    if (jz <= n && kl >= 1)
      for (int i = 1; i <= kl; ++i) AB(i - 1, jz - 1) = 0.0;
    const int lm = kl < (n - k) ? kl : (n - k);
    // first maximum of |abd(m..m+lm, k)|
    int l = m;
    double best = fabs(AB(m - 1, k - 1));
    for (int i = 1; i <= lm; ++i) {
      const double v = fabs(AB(m - 1 + i, k - 1));
      if (v > best) { best = v; l = m + i; }
    }
    pivot[k - 1] = l + k - m;
    if (fabs(AB(l - 1, k - 1)) > 1.0e-15) {
      if (l != m) {
        const double t = AB(l - 1, k - 1);
        AB(l - 1, k - 1) = AB(m - 1, k - 1);
        AB(m - 1, k - 1) = t;
      }
      const double t = -1.0 / AB(m - 1, k - 1);
      for (int i = 0; i < lm; ++i) AB(m + i, k - 1) *= t;
      int jmax = ku + pivot[k - 1];
      if (ju > jmax) jmax = ju;
      ju = jmax < n ? jmax : n;
      int mm = m, ll = l;
      for (int j = kp1; j <= ju; ++j) {
        ll -= 1;
        mm -= 1;
        const double t2 = AB(ll - 1, j - 1);
        if (ll != mm) {
          AB(ll - 1, j - 1) = AB(mm - 1, j - 1);
          AB(mm - 1, j - 1) = t2;
        }
        for (int i = 0; i < lm; ++i) AB(mm + i, j - 1) += t2 * AB(m + i, k - 1);
      }
    } else {
      info = k;
    }
  }
  pivot[n - 1] = n;
  if (fabs(AB(m - 1, n - 1)) <= 1.0e-15) info = n;
  info_all[b] = info;
}

// The same factorisation with one wave per matrix: the band is held in LDS
// (loaded and stored coalesced), every lane finds the pivot (broadcast reads),
// lanes scale the multipliers of column k and update one later column each.
// Same operations in the same order per element as k_band_factor.
__global__ __launch_bounds__(64) void k_band_factor_lds(double* __restrict__ abd_all,
                                                        int* __restrict__ piv_all,
                                                        int* __restrict__ info_all, int n, int kl,
                                                        int ku, const int* when) {
  if (when && *when == 0) return;
  extern __shared__ double sb[];  // [nrow][n]
  const int b = blockIdx.x, lane = threadIdx.x;
  const int nrow = 2 * kl + ku + 1;
  const int m = kl + ku + 1;  // 1-based diagonal row
  double* g = abd_all + (long)b * nrow * n;
  int* pivot = piv_all + (long)b * n;
#define SB(i, j) sb[(long)(i) * n + (j)]  // 0-based band row i, column j
  for (int e = lane; e < nrow * n; e += 64) sb[e] = g[e];
  __syncthreads();
  const int j0 = ku + 2, j1 = (n < m ? n : m) - 1;
  for (int jz = j0; jz <= j1; ++jz)
    for (int i = m + 1 - jz + lane; i <= kl; i += 64) SB(i - 1, jz - 1) = 0.0;
  int info = 0, jz = j1, ju = 0;
  for (int k = 1; k <= n - 1; ++k) {
    jz = jz + 1;
    __syncthreads();  // the previous step's updates are visible
    if (jz <= n)
      for (int i = lane; i < kl; i += 64) SB(i, jz - 1) = 0.0;
    __syncthreads();
    const int lm = kl < (n - k) ? kl : (n - k);
    // first maximum of |abd(m..m+lm, k)|, found by every lane
    int l = m;
    double best = fabs(SB(m - 1, k - 1));
    for (int i = 1; i <= lm; ++i) {
      const double v = fabs(SB(m - 1 + i, k - 1));
      if (v > best) {
        best = v;
        l = m + i;
      }
    }
    const int pk = l + k - m;
    if (lane == 0) pivot[k - 1] = pk;
    const double pv = SB(l - 1, k - 1), dg = SB(m - 1, k - 1);
    if (fabs(pv) > 1.0e-15) {  // uniform: every lane read the same column
      __syncthreads();         // every lane has read the column before it changes
      if (lane == 0 && l != m) {
        SB(l - 1, k - 1) = dg;
        SB(m - 1, k - 1) = pv;
      }
      __syncthreads();
      const double t = -1.0 / pv;
      for (int i = lane; i < lm; i += 64) SB(m + i, k - 1) *= t;
      int jmax = ku + pk;
      if (ju > jmax) jmax = ju;
      ju = jmax < n ? jmax : n;
      __syncthreads();  // multipliers in place
      for (int j = k + 1 + lane; j <= ju; j += 64) {
        const int ll = l - (j - k), mm = m - (j - k);
        const double t2 = SB(ll - 1, j - 1);
        if (ll != mm) {
          SB(ll - 1, j - 1) = SB(mm - 1, j - 1);
          SB(mm - 1, j - 1) = t2;
        }
        for (int i = 0; i < lm; ++i) SB(mm + i, j - 1) += t2 * SB(m + i, k - 1);
      }
    } else {
      info = k;
    }
  }
  __syncthreads();
  if (lane == 0) {
    pivot[n - 1] = n;
    if (fabs(SB(m - 1, n - 1)) <= 1.0e-15) info = n;
    info_all[b] = info;
  }
  for (int e = lane; e < nrow * n; e += 64) g[e] = sb[e];
#undef SB
}

extern "C" int mh_band_factor_gated(double* abd, int* pivot, int* info, int n, int kl, int ku,
                                    int nbatch, const int* when, void* stream) {
  if (n < 1 || kl < 0 || ku < 0 || nbatch < 1) return MH_EINVAL;
  const size_t lds = (size_t)(2 * kl + ku + 1) * n * sizeof(double);
  if (lds <= 64 * 1024) {
    hipLaunchKernelGGL(k_band_factor_lds, dim3(nbatch), dim3(64), lds, mh_stream(stream), abd,
                       pivot, info, n, kl, ku, when);
  } else {
    hipLaunchKernelGGL(k_band_factor, dim3(mh_cdiv(nbatch, 64)), dim3(64), 0, mh_stream(stream),
                       abd, pivot, info, n, kl, ku, nbatch, when);
  }
  return mh_launch_status();
}

extern "C" int mh_band_factor(double* abd, int* pivot, int* info, int n, int kl, int ku,
                              int nbatch, void* stream) {
  return mh_band_factor_gated(abd, pivot, info, n, kl, ku, nbatch, nullptr, stream);
}

// dgbsl over LDS tiles of 16 columns.  The factors are real, so the real and
// imaginary parts of a complex right-hand side are independent recurrences:
// lane 2r+c runs component c of row r, and a wave owns 32 rows.  Each tile is
// loaded (and stored) cooperatively, sixteen lanes moving one row's 256
// contiguous bytes; each lane then runs its recurrence out of LDS.  Forward
// elimination keeps b(k .. k+kl) in a register window and emits x(k-1) kl
// columns behind the input; the back substitution streams the columns
// downwards with the window x(k-m .. k-1), m = kl+ku+1, emitting x(k-1) m
// columns above the input.  Outputs replace consumed inputs in a ring of two
// tiles, stored when the tile after the next needs their slot; the forward
// result is the back substitution's input (in `sol`).  `rows` (optional) orders
// the rows by degree so that the lanes of a wave share their factors.
// In place (rhs == sol) is allowed: every tile is read before any output
// lands on it.
//
// One wave per SIMD (65 k recurrences at l_max = 255), so what a wave waits for is
// not hidden by others.  Within a tile it waits for nothing but its recurrence: the
// next tile, its row scaling and its factors and pivots (of up to eight degrees, all
// that 32 ordered rows hold) are requested before the tile is worked on, with
// unconditional clamped loads, after the stores of the tile before (a wait for the
// loads would otherwise cover the stores); and the pivots' reciprocals are formed
// when the factors are staged, so that a step of the back substitution waits for a
// product and its correction instead of a division.  The product is within 1.5 units in
// the last place (the reciprocal and itself rounded) and its remainder exact but for
// the last of 54 bits, so the corrected quotient has the division's bits unless it lies
// within about 2^-50 of the middle of two numbers; and unless the remainder is
// subnormal (right-hand sides below 2^-960), where it may be off by one unit.  28 KB of LDS at most and below 256 registers: five waves fit on a
// CU, and 1028 waves are resident at once (with 35 KB or more registers four would
// have waited for the rest: 390 us).  l_max = 255, n = 512, kl = ku = 3: 407 us ->
// 280 us (1.1 GB in four passes: 3.9 TB/s of a copy's 5.5), kl = ku = 2: 356 -> 260;
// l_max = 383, n = 97: 164 -> 119.
constexpr int kBT = 16;  // columns per tile
constexpr int kBR = 32;  // rows per wave
constexpr int kBD = 8;   // degrees per wave whose factors are staged (the first 32 rows hold 8)
constexpr int kBS = 4;   // columns whose LDS reads may be issued together (registers)

template <int KL, int KU>
__global__ __launch_bounds__(64, 2) void k_band_solve(const double* __restrict__ abd_all,
                                                   const int* __restrict__ piv_all,
                                                   const double* __restrict__ fac_row,
                                                   const double* __restrict__ fac_col,
                                                   const int* __restrict__ lm2l,
                                                   const int* __restrict__ rows,
                                                   const double2* rhs, double2* sol, int L,
                                                   int n, const int* when) {
  if (when && *when == 0) return;
  constexpr int M = KL + KU + 1;
  constexpr int NR = 2 * KL + KU + 1;
  constexpr int TP = kBT + 1;     // padded LDS row (conflict-free columns)
  constexpr int CR = 64 / kBT;    // rows per cooperative access
  constexpr int CI = kBR / CR;    // cooperative accesses per lane
  static_assert(64 % kBT == 0 && kBR % CR == 0, "cooperative tile map");
  static_assert(M <= kBT && kBD == 2 * CR, "two-tile ring, two staging accesses");
  __shared__ double2 ring[2][kBR][TP];
  // a tile's factors of the wave's degrees; row M: the pivots' reciprocals (back
  // substitution), row KL: the pivots' offsets (forward)
  __shared__ double facs[kBD][M + 1][kBT];
  const int lane = threadIdx.x;
  const int r0 = blockIdx.x * kBR;
  // this lane's row and component, and its degree's factors (lanes past the last row
  // repeat it; nothing of theirs is stored)
  const int row = lane >> 1, comp = lane & 1;
  auto row_of = [&](int r) { const int q = min(r0 + r, L - 1); return rows ? rows[q] : q; };
  const int l = lm2l[row_of(row)];
  const double* abd = abd_all + (long)l * NR * n;
  const int* pivot = piv_all + (long)l * n;
  // cooperative map: lane -> sub-row cs (rows cs + CR*it) and column cc of a tile
  const int cs = lane / kBT, cc = lane % kBT;
  int clm[CI], cl[CI];  // rows and (where a scaling wants them) their degrees
#pragma unroll
  for (int it = 0; it < CI; ++it) {
    clm[it] = row_of(cs + CR * it);
    cl[it] = fac_row || fac_col ? lm2l[clm[it]] : 0;
  }
  // the wave's distinct degrees, up to kBD: this lane's slot among them and the degrees
  // of the slots whose factors it stages (cs and cs + 4)
  int sl = 0, nd = 0, lq0 = 0, lq1 = 0;
  unsigned long long left = ~0ull;
  while (left && nd < kBD) {
    const int ld = __builtin_amdgcn_readlane(l, (int)__builtin_ctzll(left));
    const bool mine = l == ld;
    sl = mine ? nd : sl;
    if (cs >= nd) lq0 = ld;  // (slots beyond the last repeat it)
    if (cs + CR >= nd) lq1 = ld;
    left &= ~__ballot(mine);
    ++nd;
  }
  const bool fast = left == 0;  // otherwise every lane reads its factors from memory

  // (called where addresses are formed: keeps the compiler from holding the 64-bit
  // offsets of all rows in registers throughout, which would leave one wave per SIMD)
  auto fresh = [](int& i) __attribute__((always_inline)) { asm volatile("" : "+v"(i)); };

  // Q factor rows from row `row0` on, at columns base .. base + 15, four degrees an access
  auto fac_load = [&](int row0, int Q, int base, auto& v, auto& w) __attribute__((always_inline)) {
    const int c = min(max(base + cc, 0), n - 1);
    fresh(lq0), fresh(lq1);
    const double* a0 = abd_all + ((long)lq0 * NR + row0) * n + c;
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = a0[(long)q * n];
    if (nd > CR) {
      const double* a1 = abd_all + ((long)lq1 * NR + row0) * n + c;
#pragma unroll
      for (int q = 0; q < Q; ++q) w[q] = a1[(long)q * n];
    }
  };
  auto fac_put = [&](int Q, const auto& v, const auto& w) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < Q; ++q) facs[cs][q][cc] = v[q];
    if (nd > CR)
#pragma unroll
      for (int q = 0; q < Q; ++q) facs[cs + CR][q][cc] = w[q];
  };
  double2 pre[CI];  // the next tile
  double prf[CI];   // and its row scaling
  auto coop_load = [&](const double2* src, int tile, bool scale) __attribute__((always_inline)) {
    const int col = min(max(tile, 0) * kBT + cc, n - 1);
#pragma unroll
    for (int it = 0; it < CI; ++it) {
      fresh(clm[it]), fresh(cl[it]);
      pre[it] = src[(long)clm[it] * n + col];
    }
    if (scale)
#pragma unroll
      for (int it = 0; it < CI; ++it) prf[it] = fac_row[(long)cl[it] * n + col];
  };
  auto coop_put = [&](int slot, bool scale) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < CI; ++it)
      ring[slot][cs + CR * it][cc] = scale ? cscale(pre[it], prf[it]) : pre[it];
  };
  auto coop_store = [&](int tile, const double* fcol) __attribute__((always_inline)) {
    const int col = tile * kBT + cc;
#pragma unroll
    for (int it = 0; it < CI; ++it)
      if (r0 + cs + CR * it < L && col < n) {
        const double2 x = ring[tile & 1][cs + CR * it][cc];
        fresh(clm[it]), fresh(cl[it]);
        sol[(long)clm[it] * n + col] = fcol ? cscale(x, fcol[(long)cl[it] * n + col]) : x;
      }
  };
  // this lane's element of column c of the tile in a slot
  auto at = [&](int slot, int c) -> double& {
    return reinterpret_cast<double*>(&ring[slot][row][c])[comp];
  };
  const int ntile = (n + kBT - 1) / kBT;

  // ---- forward elimination: x = L^-1 P b (rows scaled by fac_row)
  if constexpr (KL > 0) {
    const bool scale = fac_row != nullptr;
    double W[KL + 1], v[KL], w[KL];
    int pv = 0, pw = 0;
#pragma unroll
    for (int j = 0; j <= KL; ++j) W[j] = 0.0;
    // iteration k (1-based): pivot swap, update of b(k+1 .. k+lmk), x(k-1) = W[0]
    // (full: an interior iteration, k <= n - KL, so every update applies; staged: the
    // factors are column c of those in LDS)
    auto iter = [&](auto full, auto staged, int k, int c) __attribute__((always_inline)) {
      constexpr bool FULL = decltype(full)::value, ST = decltype(staged)::value;
      const int lmk = FULL ? KL : min(KL, n - k);
      const int lp = (ST ? reinterpret_cast<const int*>(&facs[sl][KL][c])[0] : pivot[k - 1]) - k;
      // swap W[0] and W[lp] with selects (an indexed swap would put W in scratch)
      const double w0 = W[0];
      double p = w0;
#pragma unroll
      for (int j = 1; j <= KL; ++j) {
        const bool s = j == lp;
        p = s ? W[j] : p;
        W[j] = s ? w0 : W[j];
      }
#pragma unroll
      for (int j = 1; j <= KL; ++j)
        if (FULL || j <= lmk)
          W[j] += p * (ST ? facs[sl][j - 1][c] : abd[(long)(M + j - 1) * n + (k - 1)]);
      at(((k - 1) / kBT) & 1, (k - 1) % kBT) = p;
#pragma unroll
      for (int j = 0; j < KL; ++j) W[j] = W[j + 1];
      W[KL] = 0.0;
    };
    auto fetch = [&](int t) __attribute__((always_inline)) {
      coop_load(rhs, t, scale);
      if (fast) {
        fac_load(M, KL, t * kBT - KL, v, w);
        const int c = min(max(t * kBT - KL + cc, 0), n - 1);
        pv = piv_all[(long)lq0 * n + c];
        if (nd > CR) pw = piv_all[(long)lq1 * n + c];
      }
    };
    fetch(0);
    for (int t = 0; t < ntile; ++t) {
      const int slot = t & 1;
      __syncthreads();  // the previous tile's outputs are in the ring
      if (t >= 2) coop_store(t - 2, nullptr);
      __syncthreads();
      coop_put(slot, scale);
      if (fast) {
        fac_put(KL, v, w);
        reinterpret_cast<int*>(&facs[cs][KL][cc])[0] = pv;
        if (nd > CR) reinterpret_cast<int*>(&facs[cs + CR][KL][cc])[0] = pw;
      }
      __syncthreads();
      fetch(min(t + 1, ntile - 1));
      if (t >= 1 && (t + 1) * kBT <= n) {
        // interior tile: straight-line iterations (iteration k emits column k - 1,
        // KL behind the column that enters)
        auto tile = [&](auto staged) __attribute__((always_inline)) {
#pragma unroll
          for (int c = 0; c < kBT; ++c) {
            W[KL] = at(slot, c);
            iter(std::true_type{}, staged, t * kBT + c - KL + 1, c);
            if (c % kBS == kBS - 1) __builtin_amdgcn_sched_barrier(0);
          }
        };
        if (fast) tile(std::true_type{});
        else tile(std::false_type{});
      } else {
#pragma unroll 1
        for (int c = 0; c < kBT; ++c) {
          const int j = t * kBT + c;  // input column entering the window
          if (j >= n) break;
          W[KL] = at(slot, c);
          if (j < KL) {
            // filling: b(0 .. KL-1) move down as they arrive
#pragma unroll
            for (int q = 0; q < KL; ++q) W[q] = W[q + 1];
          } else if (fast) {
            iter(std::false_type{}, std::true_type{}, j - KL + 1, c);
          } else {
            iter(std::false_type{}, std::false_type{}, j - KL + 1, 0);
          }
        }
      }
    }
    // fewer columns than KL: finish the fill with zeros
    for (int j = n; j < KL; ++j) {
#pragma unroll
      for (int q = 0; q < KL; ++q) W[q] = W[q + 1];
      W[KL] = 0.0;
    }
    // the last iterations (nothing left to enter), then x(n-1) = W[0]
    for (int k = max(1, n - KL + 1); k <= n - 1; ++k)
      iter(std::false_type{}, std::false_type{}, k, 0);
    at(((n - 1) / kBT) & 1, (n - 1) % kBT) = W[0];
    __syncthreads();
    if (ntile > 1) coop_store(ntile - 2, nullptr);
    coop_store(ntile - 1, nullptr);
  }

  // ---- back substitution: x = U^-1 y (columns scaled by fac_col)
  {
    const double2* src = (KL > 0) ? sol : rhs;
    const bool scale = KL == 0 && fac_row;  // without a forward pass the row scaling is applied here
    double V[M], v[M], w[M];
#pragma unroll
    for (int j = 0; j < M; ++j) V[j] = 0.0;
    // iteration k (1-based, descending): finish x(k-1), update x(k-2 .. k-1-lmk)
    // (full: k > M, so every update applies)
    auto iter = [&](auto full, auto staged, int k, int c) __attribute__((always_inline)) {
      constexpr bool FULL = decltype(full)::value, ST = decltype(staged)::value;
      double x;
      if (ST) {
        const double d = facs[sl][M - 1][c], r = facs[sl][M][c], q = V[M - 1] * r;
        x = fma(fma(-q, d, V[M - 1]), r, q);
        x = fabs(q) < INFINITY ? x : q;
      } else {
        x = V[M - 1] / abd[(long)(M - 1) * n + (k - 1)];
      }
      const int lmk = FULL ? M - 1 : min(k, M) - 1;
#pragma unroll
      for (int j = 1; j < M; ++j)
        if (FULL || j <= lmk)
          V[M - 1 - j] += -x * (ST ? facs[sl][M - j - 1][c] : abd[(long)(M - j - 1) * n + (k - 1)]);
      at(((k - 1) / kBT) & 1, (k - 1) % kBT) = x;
#pragma unroll
      for (int j = M - 1; j > 0; --j) V[j] = V[j - 1];
      V[0] = 0.0;
    };
    auto fetch = [&](int u) __attribute__((always_inline)) {
      coop_load(src, u, scale);
      if (fast) fac_load(0, M, u * kBT + M, v, w);  // (u = -1: the last M steps)
    };
    // stages the factors and the pivots' reciprocals; false when a pivot is so small or
    // so large that a product with its reciprocal is not to be trusted
    auto stage = [&]() __attribute__((always_inline)) {
      auto usable = [](double d) { return fabs(d) > 0x1p-900 && fabs(d) < 0x1p900; };
      fac_put(M, v, w);
      bool ok = usable(v[M - 1]);
      facs[cs][M][cc] = 1.0 / v[M - 1];
      if (nd > CR) {
        ok = ok && usable(w[M - 1]);
        facs[cs + CR][M][cc] = 1.0 / w[M - 1];
      }
      return (bool)__all(ok);
    };
    bool st = false;
    fetch(ntile - 1);
    for (int u = ntile - 1; u >= 0; --u) {
      const int slot = u & 1;
      __syncthreads();  // the previous tile's outputs are in the ring
      if (u + 2 < ntile) coop_store(u + 2, fac_col);
      __syncthreads();
      coop_put(slot, scale);
      if (fast) st = stage();
      __syncthreads();
      fetch(u - 1);
      if ((u + 1) * kBT + M <= n) {
        // interior tile: straight-line iterations (k = column + M + 1 <= n, k > M)
        auto tile = [&](auto staged) __attribute__((always_inline)) {
#pragma unroll
          for (int c = kBT - 1; c >= 0; --c) {
            const double y = at(slot, c);
            iter(std::true_type{}, staged, u * kBT + c + M + 1, c);
            V[0] = y;
            if (c % kBS == 0) __builtin_amdgcn_sched_barrier(0);
          }
        };
        if (st) tile(std::true_type{});
        else tile(std::false_type{});
      } else {
#pragma unroll 1
        for (int c = kBT - 1; c >= 0; --c) {
          const int col = u * kBT + c;  // input column entering the window from below
          if (col >= n) continue;
          const double y = at(slot, c);
          const int k = col + M + 1;
          if (k <= n) {
            if (st) iter(std::false_type{}, std::true_type{}, k, c);
            else iter(std::false_type{}, std::false_type{}, k, 0);
            V[0] = y;
          } else {
            // initial fill of x(n-1) .. x(n-M), by distance from the top
            const int pos = M - 1 - (n - 1 - col);
#pragma unroll
            for (int j = 0; j < M; ++j)
              if (j == pos) V[j] = y;
          }
        }
      }
    }
    __syncthreads();
    if (fast) st = stage();
    __syncthreads();
    for (int k = min(M, n); k >= 1; --k)
      if (st) iter(std::false_type{}, std::true_type{}, k, kBT - 1 - M + k);
      else iter(std::false_type{}, std::false_type{}, k, 0);
    __syncthreads();
    if (ntile > 1) coop_store(1, fac_col);
    coop_store(0, fac_col);
  }
}

extern "C" int mh_band_solve_gated(const double* abd, const int* pivot, const double* fac_row,
                                   const double* fac_col, const int* lm2l, const int* rows,
                                   const double* rhs, double* sol, int L, int n, int kl, int ku,
                                   const int* when, void* stream) {
  if (L < 1 || n < 1 || kl < 0 || ku < 0 || kl > 4 || ku > 4) return MH_EINVAL;
  const dim3 g(mh_cdiv(L, kBR)), blk(64);  // one wave of 32 rows (two lanes each) per workgroup
  hipStream_t st = mh_stream(stream);
  const double2* r = reinterpret_cast<const double2*>(rhs);
  double2* o = reinterpret_cast<double2*>(sol);
#define MH_BAND_CASE(A, B)                                                                      \
  if (kl == A && ku == B) {                                                                     \
    hipLaunchKernelGGL((k_band_solve<A, B>), g, blk, 0, st, abd, pivot, fac_row, fac_col, lm2l, \
                       rows, r, o, L, n, when);                                                 \
    return mh_launch_status();                                                                  \
  }
#define MH_BAND_ROW(A) MH_BAND_CASE(A, 0) MH_BAND_CASE(A, 1) MH_BAND_CASE(A, 2) MH_BAND_CASE(A, 3) MH_BAND_CASE(A, 4)
  MH_BAND_ROW(0) MH_BAND_ROW(1) MH_BAND_ROW(2) MH_BAND_ROW(3) MH_BAND_ROW(4)
#undef MH_BAND_ROW
#undef MH_BAND_CASE
  return MH_EINVAL;
}

extern "C" int mh_band_solve(const double* abd, const int* pivot, const double* fac_row,
                             const double* fac_col, const int* lm2l, const int* rows,
                             const double* rhs, double* sol, int L, int n, int kl, int ku,
                             void* stream) {
  return mh_band_solve_gated(abd, pivot, fac_row, fac_col, lm2l, rows, rhs, sol, L, n, kl, ku,
                             nullptr, stream);
}
