// Azimuthal real FFTs between Fourier buffers F[c][m][t][b] (complex, m < n_m)
// and grid rows G[c][b][t][phi] (real, n_phi = 2*Mh points), norm="forward"
// (the inverse carries no scale, the forward scales by 1/n_phi).
//
// A real transform of length 2*Mh is done as one complex Stockham FFT of
// length Mh with the standard even/odd packing.  One workgroup handles RB
// consecutive batch rows b of one (component, theta) pair: it reads or writes F
// in RB-wide contiguous complex runs (128 bytes for the usual eight) and packs or
// unpacks the conjugate pairs on the way, which transposes the rows through LDS.
// The transform itself belongs to LPR lanes of one wave per row: radix 8 and 9
// passes in registers, exchanged through the row's LDS in place (a wave's LDS
// accesses execute in order), without workgroup barriers; the first pass of the
// forward and the last of the inverse transform access G directly.  So a row
// crosses LDS three times at Mh = 576 (9 x 8 x 8) and twice at 192, and the only
// barrier is the one between the transposition and the passes.
//
// What bounds it is HBM and the latency of one block's rows: l_max = 383, 97
// columns move 0.86 GB in 249 us (inverse) and 200 us (forward), 3.5 and 4.3 TB/s,
// where workgroup-wide radix-4 passes with a barrier each took 622 us; l_max = 127,
// 3 x 65 columns 50 and 41 us (112 and 95).
#include "fft_lds.h"

typedef MhFftArgs FftArgs;
#define TW(a) reinterpret_cast<const double2*>((a).tw)
#define TW2(a) reinterpret_cast<const double2*>((a).tw2)

__device__ __forceinline__ double2* fft_lds(double2* b0, double2* b1, const FftArgs& a, double dir) {
  return fft_lds_rows(b0, b1, a.Mh, a.nstage, a.radix, a.RB, TW(a), dir);
}

// ---------------------------------------------------------------- in-wave transforms

namespace {

// Plan of the in-wave transform of length Mh.
struct WPlan {
  int nst, radix[10];
  unsigned magic[10];  // ceil(2^32 / Ns) of each pass: x / Ns = umulhi(x, magic), x < 2^16
  int lsh, lpr;        // lanes per row (a power of two)
  int rsh, RB;         // rows per workgroup (a power of two; taken from the argument)
  int S;               // LDS row stride (complex values)
  int psh;             // padding: element i of a row sits at i + (i >> psh)
};

constexpr WPlan make_wplan(int Mh) {
  WPlan p{};
  if (Mh < 2 || Mh > 768) return p;
  // about 12 elements per lane (registers)
  p.lsh = 1;
  while (p.lsh < 6 && (12 << p.lsh) < Mh) ++p.lsh;
  p.lpr = 1 << p.lsh;
  int n = Mh, k = 0;
  // odd radices first: the first pass writes R consecutive elements per lane,
  // free of bank conflicts at an odd stride; 9 where one pass of the lanes holds it
  while (n % 9 == 0 && Mh / 9 <= p.lpr) { p.radix[k++] = 9; n /= 9; }
  while (n % 5 == 0) { p.radix[k++] = 5; n /= 5; }
  while (n % 3 == 0) { p.radix[k++] = 3; n /= 3; }
  while (n % 8 == 0) { p.radix[k++] = 8; n /= 8; }
  if (n == 4) { p.radix[k++] = 4; n = 1; }
  if (n == 2) { p.radix[k++] = 2; n = 1; }
  if (n != 1) return p;
  long Ns = 1;
  for (int s = 0; s < k; ++s) {
    p.magic[s] = Ns > 1 ? (unsigned)(((1ull << 32) + Ns - 1) / Ns) : 0u;
    Ns *= p.radix[s];
  }
  p.psh = p.radix[0] % 2 ? 30 : 3;
  // a row stride of 8 (mod 16) complex values: the 8 x 8 transposition and the
  // passes of several rows per wave spread over all banks
  const int row = Mh + (Mh >> p.psh);
  p.S = row + ((8 - row) % 16 + 16) % 16;
  // eight rows (128-byte runs of F), more where rows are so short that a
  // workgroup would have fewer than four waves
  p.rsh = 3;
  while (p.rsh < 5 && (p.lpr << p.rsh) < 256) ++p.rsh;
  while (((long)p.S << p.rsh) * 16 > 80 * 1024) --p.rsh;
  p.RB = 1 << p.rsh;
  p.nst = k;
  return p;
}

// Lengths with a compiled plan; others run the same passes with the plan as an
// argument.
#define MH_WFFT_COMPILED(X) \
  X(24) X(48) X(64) X(96) X(128) X(192) X(256) X(288) X(384) X(512) X(576) X(768)

constexpr bool wave_compiled(int Mh) {
  switch (Mh) {
#define MH_WC(V) case V:
    MH_WFFT_COMPILED(MH_WC)
#undef MH_WC
    return true;
    default: return false;
  }
}

// Whether rows of length Mh are transformed by single waves: compiled plans, and run-time
// plans from 100 on or, without a factor 5, from 50 on.  Shorter rows are a few elements a
// lane, and the run-time passes' index arithmetic costs more than the workgroup's
// barriers that they save; radix 9 and 8 save a pass or two at 54 and 72, radix 5 none
// (k_fft_inverse -> k_wfft_inverse, 8 columns: 30 5.7 -> 7.5 us, 36 6.0 -> 6.6, 60 7.3 -> 7.5, 80
// 8.3 -> 9.0, 90 10.0 -> 10.4; 54 8.3 -> 7.5, 72 9.1 -> 7.0, 100 9.9 -> 8.0, 120 12.0 -> 7.8).
constexpr bool wave_rows(int Mh) {
  if (wave_compiled(Mh)) return true;
  return (Mh >= 100 || (Mh >= 50 && Mh % 5 != 0)) && make_wplan(Mh).nst > 0;
}

// Geometry and plan of a launch: compile-time constants when MH > 0.
template <int MH>
struct WGeo {
  static constexpr WPlan P = make_wplan(MH);
  __device__ static const WPlan& plan(const WPlan&) { return P; }
};
template <>
struct WGeo<0> {
  __device__ static const WPlan& plan(const WPlan& p) { return p; }
};

__device__ __forceinline__ void wave_fence() {
  // other lanes of the wave read what this lane wrote: order the LDS accesses
  // (the hardware executes a wave's LDS instructions in order)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Work of this workgroup.  Consecutive row blocks of one latitude and consecutive
// latitudes share 128-byte lines of F, so each XCD (workgroups i and i + 8) gets a
// contiguous range of them.
__device__ __forceinline__ bool wfft_block(const FftArgs& a, int RB, int& c, int& t, int& bs) {
  const int nx = (a.B + RB - 1) / RB, n = nx * a.T * a.ncomp, per = (n + 7) / 8;
  const int L = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || L >= n) return false;
  const int ct = L / nx;
  bs = (L - ct * nx) * RB;
  c = ct / a.T;
  t = ct - c * a.T;
  return true;
}

// One pass of radix R over a row: butterflies li + q lpr (q < NQ), element e
// read by ld(e) and written by st(e, v).
template <int R, int NQ, typename Ld, typename St>
__device__ __forceinline__ void wave_pass(int lpr, int Mh, int Ns, unsigned magic, int li,
                                          const double2* __restrict__ tw, double dir, Ld ld, St st) {
  const int nb = Mh / R, tstep = nb / Ns;
  double2 v[NQ][R];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (q * lpr < nb) {  // uniform
      const int bf = li + q * lpr;
      if (bf < nb)
#pragma unroll
        for (int r = 0; r < R; ++r) v[q][r] = ld(bf + r * nb);
    }
  }
  wave_fence();
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (q * lpr < nb) {
      const int bf = li + q * lpr;
      const int g = Ns > 1 ? (int)__umulhi((unsigned)bf, magic) : bf, k = bf - g * Ns;
      if (bf < nb) {
        if (Ns > 1) {
          // exp(-+ 2 pi i k r / (Ns R)) from the table at r = 1, 2, 4 and products
          auto get = [&](int r) {
            double2 w = tw[r * k * tstep];
            w.y *= -dir;
            return w;
          };
          const double2 w1 = get(1);
          v[q][1] = cmul(v[q][1], w1);
          if constexpr (R > 2) {
            const double2 w2 = get(2);
            v[q][2] = cmul(v[q][2], w2);
            if constexpr (R > 3) {
              const double2 w3 = cmul(w1, w2);
              v[q][3] = cmul(v[q][3], w3);
              if constexpr (R > 4) {
                const double2 w4 = get(4);
                v[q][4] = cmul(v[q][4], w4);
                if constexpr (R > 5) {
                  v[q][5] = cmul(v[q][5], cmul(w1, w4));
                  v[q][6] = cmul(v[q][6], cmul(w2, w4));
                  v[q][7] = cmul(v[q][7], cmul(w3, w4));
                  if constexpr (R > 8) v[q][8] = cmul(v[q][8], cmul(w4, w4));
                }
              }
            }
          }
        }
        dft_any<R>(v[q], dir);
#pragma unroll
        for (int r = 0; r < R; ++r) st(g * Ns * R + k + r * Ns, v[q][r]);
      }
    }
  }
  wave_fence();
}

// Pass s of the run-time plan (rounds for at most 12 elements per lane, a butterfly
// more where the radix does not divide them).
template <typename Ld, typename St>
__device__ __forceinline__ void wave_pass_rt(const WPlan& p, int s, int Mh, int Ns, int li,
                                             const double2* __restrict__ tw, double dir, Ld ld,
                                             St st) {
  const unsigned mg = p.magic[s];
  switch (p.radix[s]) {
    case 8: wave_pass<8, 2>(p.lpr, Mh, Ns, mg, li, tw, dir, ld, st); break;
    case 9: wave_pass<9, 1>(p.lpr, Mh, Ns, mg, li, tw, dir, ld, st); break;
    case 4: wave_pass<4, 3>(p.lpr, Mh, Ns, mg, li, tw, dir, ld, st); break;
    case 5: wave_pass<5, 3>(p.lpr, Mh, Ns, mg, li, tw, dir, ld, st); break;
    case 3: wave_pass<3, 4>(p.lpr, Mh, Ns, mg, li, tw, dir, ld, st); break;
    default: wave_pass<2, 6>(p.lpr, Mh, Ns, mg, li, tw, dir, ld, st); break;
  }
}

// All passes of a row: the first reads by ld0, the last writes by stN, the others
// exchange through the row by ld, st.
template <int MH, int S, int NS, typename L0, typename Ld, typename St, typename Sn>
__device__ __forceinline__ void wave_passes_ct(int li, const double2* __restrict__ tw, double dir,
                                               L0 ld0, Ld ld, St st, Sn stN) {
  constexpr WPlan P = make_wplan(MH);
  if constexpr (S < P.nst) {
    constexpr int R = P.radix[S], NQ = (MH / R + P.lpr - 1) / P.lpr;
    constexpr bool first = S == 0, last = S == P.nst - 1;
    if constexpr (first && last) wave_pass<R, NQ>(P.lpr, MH, NS, P.magic[S], li, tw, dir, ld0, stN);
    else if constexpr (first) wave_pass<R, NQ>(P.lpr, MH, NS, P.magic[S], li, tw, dir, ld0, st);
    else if constexpr (last) wave_pass<R, NQ>(P.lpr, MH, NS, P.magic[S], li, tw, dir, ld, stN);
    else wave_pass<R, NQ>(P.lpr, MH, NS, P.magic[S], li, tw, dir, ld, st);
    wave_passes_ct<MH, S + 1, NS * R>(li, tw, dir, ld0, ld, st, stN);
  }
}

}  // namespace

// F -> G as k_fft_inverse below.
template <int MH>
__global__ __launch_bounds__(512, MH > 0 ? 4 : 2) void k_wfft_inverse(FftArgs a, WPlan pa) {
  extern __shared__ double2 lds[];
  const WPlan& p = WGeo<MH>::plan(pa);
  int c, t, bs;
  const int RB = pa.RB, rsh = pa.rsh;
  if (!wfft_block(a, RB, c, t, bs)) return;  // uniform per workgroup
  const int Mh = MH > 0 ? MH : a.Mh, M = a.n_m, nrow = min(RB, a.B - bs);
  const double2* tw = TW(a);
  const double2* tw2 = TW2(a);
  const double* Fct = a.F + c * a.Fc_stride + (long)t * 2 * a.FB + 2L * bs;
  // packed spectrum by conjugate pairs (pair q, row j): Z_q = E + iO and Z_{Mh-q} =
  // conj(E) + i conj(O), E = X_q + conj(X_{Mh-q}), O = (X_q - conj(X_{Mh-q})) e^{+2 pi i q/n}
  constexpr int U = 3;
  const int np = (Mh / 2 + 1) << rsh, nth = blockDim.x;
  for (int e0 = threadIdx.x; e0 < np; e0 += U * nth) {
    double2 x[U], y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + u * nth, q = e >> rsh, j = e & (RB - 1);
      x[u] = y[u] = make_double2(0.0, 0.0);
      if (e < np && j < nrow) {
        if (q < M) x[u] = *reinterpret_cast<const double2*>(Fct + (long)q * a.Fm_stride + 2 * j);
        if (q > 0 && Mh - q < M)
          y[u] = *reinterpret_cast<const double2*>(Fct + (long)(Mh - q) * a.Fm_stride + 2 * j);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = e0 + u * nth, q = e >> rsh, j = e & (RB - 1);
      if (e < np) {
        if (q == 0) x[u].y = 0.0;
        const double2 yc = cconj(y[u]);
        const double2 E = cadd(x[u], yc), O = cmul(csub(x[u], yc), cconj(tw2[q]));
        double2* row = lds + j * p.S;
        row[q + (q >> p.psh)] = make_double2(E.x - O.y, E.y + O.x);
        const int qc = Mh - q;
        if (q > 0 && qc > q) row[qc + (qc >> p.psh)] = make_double2(E.x + O.y, O.x - E.y);
      }
    }
  }
  __syncthreads();
  const int j = threadIdx.x >> p.lsh, li = threadIdx.x & (p.lpr - 1);
  if (j >= nrow) return;  // rows past the batch
  double2* row = lds + j * p.S;
  double2* G = reinterpret_cast<double2*>(a.G + c * a.Gc_stride + ((long)(bs + j) * a.T + t) * 2L * Mh);
  auto ld = [&](int e) { return row[e + (e >> p.psh)]; };
  auto st = [&](int e, double2 v) { row[e + (e >> p.psh)] = v; };
  auto out = [&](int e, double2 v) { G[e] = v; };
  if constexpr (MH > 0) {
    wave_passes_ct<MH, 0, 1>(li, tw, 1.0, ld, ld, st, out);
  } else {
    int Ns = 1;
    for (int s = 0; s + 1 < p.nst; ++s) {
      wave_pass_rt(p, s, Mh, Ns, li, tw, 1.0, ld, st);
      Ns *= p.radix[s];
    }
    wave_pass_rt(p, p.nst - 1, Mh, Ns, li, tw, 1.0, ld, out);
  }
}

// G -> F as k_fft_forward below.
template <int MH>
__global__ __launch_bounds__(512, MH > 0 ? 4 : 2) void k_wfft_forward(FftArgs a, WPlan pa) {
  extern __shared__ double2 lds[];
  const WPlan& p = WGeo<MH>::plan(pa);
  int c, t, bs;
  const int RB = pa.RB, rsh = pa.rsh;
  if (!wfft_block(a, RB, c, t, bs)) return;  // uniform per workgroup
  const int Mh = MH > 0 ? MH : a.Mh, M = a.n_m, nrow = min(RB, a.B - bs);
  const double2* tw = TW(a);
  const double2* tw2 = TW2(a);
  {
    const int j = threadIdx.x >> p.lsh, li = threadIdx.x & (p.lpr - 1);
    // (the compiled plans work on the first row again instead of branching around the
    // passes: l_max = 383, 97 columns 198 against 207 us)
    if (j < (MH > 0 ? RB : nrow)) {
      double2* row = lds + j * p.S;
      const double2* G = reinterpret_cast<const double2*>(
          a.G + c * a.Gc_stride + ((long)(bs + (j < nrow ? j : 0)) * a.T + t) * 2L * Mh);
      auto in = [&](int e) { return G[e]; };
      auto ld = [&](int e) { return row[e + (e >> p.psh)]; };
      auto st = [&](int e, double2 v) { row[e + (e >> p.psh)] = v; };
      if constexpr (MH > 0) {
        wave_passes_ct<MH, 0, 1>(li, tw, -1.0, in, ld, st, st);
      } else {
        wave_pass_rt(p, 0, Mh, 1, li, tw, -1.0, in, st);
        int Ns = p.radix[0];
        for (int s = 1; s < p.nst; ++s) {
          wave_pass_rt(p, s, Mh, Ns, li, tw, -1.0, ld, st);
          Ns *= p.radix[s];
        }
      }
    }
  }
  __syncthreads();
  double scale = 1.0 / (2.0 * Mh);
  if (a.comp_scale && a.comp_scale[c]) scale *= a.ost2[t];
  double* Fct = a.F + c * a.Fc_stride + (long)t * 2 * a.FB + 2L * bs;
  // X_q = E + w O and X_{Mh-q} = conj(E - w O), w = e^{-2 pi i q/n}, by pairs
  const int np = (Mh / 2 + 1) << rsh;
  for (int e = threadIdx.x; e < np; e += blockDim.x) {
    const int q = e >> rsh, j = e & (RB - 1), qc = q == 0 ? 0 : Mh - q;
    if (j >= nrow) continue;
    const double2* row = lds + j * p.S;
    const double2 Z = row[q + (q >> p.psh)], Zc = cconj(row[qc + (qc >> p.psh)]);
    const double2 E = cscale(cadd(Z, Zc), 0.5);
    const double2 D = csub(Z, Zc);
    const double2 O = cmul(tw2[q], make_double2(0.5 * D.y, -0.5 * D.x));  // w (Z - Zc) / (2i)
    if (q < M)
      *reinterpret_cast<double2*>(Fct + (long)q * a.Fm_stride + 2 * j) = cscale(cadd(E, O), scale);
    if (qc > q && qc < M)
      *reinterpret_cast<double2*>(Fct + (long)qc * a.Fm_stride + 2 * j) =
          cscale(cconj(csub(E, O)), scale);
  }
}

template <int MH>
static void wfft_launch(int forward, const FftArgs& a, const WPlan& p, hipStream_t st) {
  const size_t bytes = (size_t)p.RB * p.S * sizeof(double2);
  const long n = (long)mh_cdiv(a.B, p.RB) * a.T * a.ncomp;
  const dim3 grid((unsigned)((n + 7) / 8 * 8)), blk(mh_cdiv(p.RB * p.lpr, 64) * 64);
  if (forward) hipLaunchKernelGGL((k_wfft_forward<MH>), grid, blk, bytes, st, a, p);
  else hipLaunchKernelGGL((k_wfft_inverse<MH>), grid, blk, bytes, st, a, p);
}

// ---------------------------------------------------------------- workgroup rows
// Workgroup-wide transforms for the rows that do not fit a wave's registers and for
// short rows without a compiled plan (wave_rows()).

// F (spectral) -> G (grid): x_j = sum_k X_k e^{+2 pi i jk/n}, X_{n-k} = conj(X_k).
__global__ __launch_bounds__(256) void k_fft_inverse(FftArgs a) {
  extern __shared__ double2 lds[];
  double2* b0 = lds;
  double2* b1 = lds + a.RB * a.Mh;
  const int c = blockIdx.z, t = blockIdx.y, bs = blockIdx.x * a.RB;
  const int Mh = a.Mh;
  const double* Fct = a.F + c * a.Fc_stride + (long)t * 2 * a.FB;
  for (int idx = threadIdx.x; idx < a.RB * Mh; idx += blockDim.x) {
    const int m = idx / a.RB, j = idx - m * a.RB;
    double2 v = make_double2(0.0, 0.0);
    if (m < a.n_m && bs + j < a.B) {
      const double* src = Fct + (long)m * a.Fm_stride + 2L * (bs + j);
      v = make_double2(src[0], m == 0 ? 0.0 : src[1]);
    }
    b0[j * Mh + m] = v;
  }
  __syncthreads();
  // Z_k = E_k + i O_k,  E_k = X_k + conj(X_{Mh-k}),  O_k = (X_k - conj(X_{Mh-k})) e^{+2 pi i k/n}
  for (int idx = threadIdx.x; idx < a.RB * Mh; idx += blockDim.x) {
    const int j = idx / Mh, k = idx - j * Mh;
    const double2 X = b0[j * Mh + k];
    const double2 Xc = (k == 0) ? make_double2(0.0, 0.0) : cconj(b0[j * Mh + Mh - k]);
    const double2 E = cadd(X, Xc);
    const double2 O = cmul(csub(X, Xc), cconj(TW2(a)[k]));
    b1[j * Mh + k] = make_double2(E.x - O.y, E.y + O.x);
  }
  __syncthreads();
  double2* res = fft_lds(b1, b0, a, 1.0);
  for (int idx = threadIdx.x; idx < a.RB * Mh; idx += blockDim.x) {
    const int j = idx / Mh, q = idx - j * Mh;
    if (bs + j < a.B) {
      double2* dst = reinterpret_cast<double2*>(a.G + c * a.Gc_stride +
                                                ((long)(bs + j) * a.T + t) * 2L * Mh);
      dst[q] = res[j * Mh + q];
    }
  }
}

// G (grid) -> F (spectral), X_k = (1/n) sum_j x_j e^{-2 pi i jk/n}, k < n_m,
// optionally times ost2[t] per component.
__global__ __launch_bounds__(256) void k_fft_forward(FftArgs a) {
  extern __shared__ double2 lds[];
  double2* b0 = lds;
  double2* b1 = lds + a.RB * a.Mh;
  const int c = blockIdx.z, t = blockIdx.y, bs = blockIdx.x * a.RB;
  const int Mh = a.Mh;
  for (int idx = threadIdx.x; idx < a.RB * Mh; idx += blockDim.x) {
    const int j = idx / Mh, q = idx - j * Mh;
    double2 v = make_double2(0.0, 0.0);
    if (bs + j < a.B) {
      const double2* src = reinterpret_cast<const double2*>(
          a.G + c * a.Gc_stride + ((long)(bs + j) * a.T + t) * 2L * Mh);
      v = src[q];
    }
    b0[j * Mh + q] = v;
  }
  __syncthreads();
  double2* res = fft_lds(b0, b1, a, -1.0);
  double scale = 1.0 / (2.0 * Mh);
  if (a.comp_scale && a.comp_scale[c]) scale *= a.ost2[t];
  double* Fct = a.F + c * a.Fc_stride + (long)t * 2 * a.FB;
  for (int idx = threadIdx.x; idx < a.RB * a.n_m; idx += blockDim.x) {
    const int m = idx / a.RB, j = idx - m * a.RB;
    if (bs + j >= a.B) continue;
    const double2 Z = res[j * Mh + m];
    const double2 Zc = cconj(res[j * Mh + ((Mh - m) % Mh)]);
    const double2 E = cscale(cadd(Z, Zc), 0.5);
    const double2 D = csub(Z, Zc);
    const double2 O = make_double2(0.5 * D.y, -0.5 * D.x);  // (Z - Zc) / (2i)
    const double2 X = cadd(E, cmul(TW2(a)[m], O));
    double* dst = Fct + (long)m * a.Fm_stride + 2L * (bs + j);
    dst[0] = X.x * scale;
    dst[1] = X.y * scale;
  }
}

extern "C" int mh_fft(int forward, const MhFftArgs* args, void* stream) {
  const FftArgs& a = *args;
  if (a.Mh < 2 || a.RB < 1 || a.B < 1 || a.T < 1 || a.ncomp < 1 || a.n_m > a.Mh) return MH_EINVAL;
  int prod = 1;
  for (int s = 0; s < a.nstage; ++s) {
    const int R = a.radix[s];
    if (R != 2 && R != 3 && R != 4 && R != 5) return MH_EINVAL;
    prod *= R;
  }
  if (prod != a.Mh) return MH_EINVAL;
  const size_t lds = 2ull * a.RB * a.Mh * sizeof(double2);
  if (lds > 160 * 1024) return MH_EINVAL;
  if (wave_rows(a.Mh)) {
    if ((long)a.B * a.T * a.ncomp >= 0x7fffffffL) return MH_EINVAL;
    WPlan p = make_wplan(a.Mh);
    while (p.rsh > 0 && (p.RB >> 1) >= a.B) p.RB = 1 << --p.rsh;  // no rows past a short batch
    // the run-time passes take 159 registers, so that a workgroup of eight whole waves is
    // alone on its CU: four rows there (Mh = 400: 9 columns 41 -> 25 us, 97 229 -> 175 inverse
    // and 204 -> 152 forward; compiled plans lose up to 9 % of the forward transform to
    // the shorter runs of F)
    if (!wave_compiled(a.Mh) && p.lsh == 6 && p.rsh > 2) p.RB = 1 << (p.rsh = 2);
    switch (a.Mh) {
#define MH_WCASE(V) case V: wfft_launch<V>(forward, a, p, mh_stream(stream)); break;
      MH_WFFT_COMPILED(MH_WCASE)
#undef MH_WCASE
      default: wfft_launch<0>(forward, a, p, mh_stream(stream));
    }
    return mh_launch_status();
  }
  dim3 grid(mh_cdiv(a.B, a.RB), a.T, a.ncomp);
  if (forward)
    hipLaunchKernelGGL(k_fft_forward, grid, dim3(256), lds, mh_stream(stream), a);
  else
    hipLaunchKernelGGL(k_fft_inverse, grid, dim3(256), lds, mh_stream(stream), a);
  return mh_launch_status();
}

