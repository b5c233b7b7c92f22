// FP64 Legendre synthesis and analysis for gfx950 (16x16x4 FP64 MFMA).
//
// Vector fields are handled in their sin(theta)-weighted form with the P_lm
// tables alone.  With c_l = sqrt((l^2 - m^2) / (4 l^2 - 1)),
//   sin(theta) dP_l/dtheta = l c_{l+1} P_{l+1} - (l + 1) c_l P_{l-1},
// so the theta and phi components of a (Q, S, T) group are scalar syntheses of
//   V_l = (l - 1) c_l S_{l-1} - (l + 2) c_{l+1} S_{l+1} + i m T_l
//   W_l = i m S_l - (l - 1) c_l T_{l-1} + (l + 2) c_{l+1} T_{l+1}
// over l = m .. l_max + 1, and the analysis of a pair (f_theta, f_phi) takes
// the scalar sums A_l of both up to l_max + 1 and combines neighbours:
//   l(l+1) S_l =  l c_{l+1} A_{l+1}(f_theta) - (l+1) c_l A_{l-1}(f_theta) - i m A_l(f_phi)
//   l(l+1) T_l = -l c_{l+1} A_{l+1}(f_phi)   + (l+1) c_l A_{l-1}(f_phi)   - i m A_l(f_theta).
// That is three products per group and theta pair instead of five (P Q, P T,
// P S, dP S, dP T), and two per pair instead of four; a workgroup takes both
// parities of l - m, so each input is read once for both.
//
// Tables: syn[m][p][k][j] and ana[m][p][j][k] (legendre.hip) with the degrees
// up to l_max + 1; `lcf` holds (l - 1) c_l, (l + 2) c_{l+1}, (l + 1) c_l and l c_{l+1}
// for the rows lm_start[m] + mi + (l - m).
//
// What bounds the kernels besides the matrix units is vector instructions: an
// FP64 MFMA takes 64 cycles of its SIMD and every FP64 or address instruction of
// the staging competes for issue.  So all addresses are a scalar base plus a
// lane offset that stays fixed or grows by one addition a chunk, and rows
// before the first degree, past the last one or past the batch are read through
// buffer descriptors that return zero there, without compares or selects.
#include <algorithm>
#include <type_traits>

#include "legendre_common.h"

namespace {

// Descriptor of `bytes` bytes at the (uniform) address p; reads past them give 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t brsrc(const double* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(p), 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ double2 bld2(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
constexpr unsigned kOut = 0x80000000u;  // an offset past every descriptor
// The same for rows that 32-bit offsets do not reach: row i < n of `ld` bytes.
__device__ __forceinline__ double2 gld2(const double* p, int i, int n, long ld, int b, int B) {
  if (i < 0 || i >= n || b >= B) return make_double2(0.0, 0.0);
  return *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(p) + i * ld + 16L * b);
}
constexpr int kAnaWindow = 60;          // degree indices per entry of the analysis work list

// The neighbour combination of the vector analysis for element v of parity p: `opp`
// the other parity's sums of this lane, `same` the other field's of this parity, cl =
// ((l + 1) c_l, l c_{l+1}).  S = l c_{l+1} A_{l+1} - (l + 1) c_l A_{l-1} - i m B_l, and T the first
// two negated (sgn).
__device__ __forceinline__ double ana_combine(const double4_t& opp, double same, int p, int v, double sgn,
                                              double2 cl, double dm, int lane) {
  // A_{l-1} and A_{l+1}: the other parity at k - 1, k (p = 0) or k, k + 1 (p = 1); a
  // neighbouring k is the next lane group's element, or the next element of the
  // group at the other end
  const int g = lane >> 4;  // accumulator row of element v: g + 4 v
  const double here = opp[v];
  double am, ap;
  if (p == 0) {
    const double give = g == 3 ? (v > 0 ? opp[v > 0 ? v - 1 : 0] : 0.0) : here;
    am = __shfl(give, (lane + 48) & 63);
    ap = here;
  } else {
    const double give = g == 0 ? (v < 3 ? opp[v < 3 ? v + 1 : 3] : 0.0) : here;
    ap = __shfl(give, (lane + 16) & 63);
    am = here;
  }
  return fma(sgn * cl.y, ap, fma(-sgn * cl.x, am, imul_pair(same, -dm, lane)));
}

}  // namespace

// ---------------------------------------------------------------- synthesis
// One workgroup of four waves: order m, 2 NT tiles of 16 theta pairs, both
// parities, and three column tiles of 8 complex columns that share every table
// operand: the three components of 8 columns of one group (VEC), or 8 NF
// columns of a scalar group.  A wave takes one parity of NT tiles, so the four
// SIMDs have equal shares whatever the number of tiles; the parities meet in
// LDS at the end (the even wave stores the northern rows, the odd one the
// southern).  The input tile of CH consecutive degrees is combined once and
// staged in LDS by parity (double-buffered, one barrier a chunk); the next
// chunk's inputs are requested before the current chunk's MFMAs, and each table
// operand is refilled for the next chunk right after its use, so that every
// load has a whole chunk (4 x NT x NF MFMAs) to arrive.  BIG: rows past the reach of
// the descriptors' offsets, with addresses and compares per load.
template <bool VEC, int NF, int NT, bool BIG = false>
__global__ __launch_bounds__(256, NT == 3 && NF == 3 ? 2 : 3) void k_syn64(SynArgs a, int n_m) {
  constexpr int CH = 32, SPC = CH / 8;  // degrees and MFMA steps (per parity) of a chunk
  constexpr int NS = VEC ? 1 : NF;      // scalar column tiles staged per item
  constexpr int CW = VEC ? 8 : 8 * NF;  // complex columns per workgroup
  constexpr int XS = 2 * NF * CH * 16, EX = 4 * NT * 256;
  __shared__ double smem[XS > EX ? XS : EX];
  double(*const xs)[NF][CH][16] = reinterpret_cast<double(*)[NF][CH][16]>(smem);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nxg = (a.B + CW - 1) / CW, nx = a.ngroups * nxg;
  const int nt = (a.H + 15) / 16, ny = (nt + 2 * NT - 1) / (2 * NT);
  // XCD-aware order: all tiles of one m on one XCD (workgroups b and b + 8), the
  // theta tiles of one column block next to each other, so that the inputs and
  // the order's table are read into that XCD's L2 once
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int m = (slot / (nx * ny)) * 8 + xcd;
  if (m >= n_m) return;  // uniform per workgroup
  const int mo = m * (a.minc > 1 ? a.minc : 1);
  const int rem = slot % (nx * ny), tx = rem / ny, ty = rem - tx * ny;
  const int g = tx / nxg, bc0 = (tx - g * nxg) * CW;  // group, first column in it
  const int par = w & 1, t0w = ty * 2 * NT + (w >> 1) * NT;  // parity, first tile of the wave
  const int col = lane & 15, kk = lane >> 4;
  const long lms = a.lm_start[m];
  const int n = a.l_max + 1 - mo;  // degrees of the order
  const int n1 = VEC ? n + 1 : n;  // rows of the sums
  const double dm = (double)mo;
  // staging item of this thread: degree row r of the chunk, complex column cc
  const int r = threadIdx.x >> 3, cc = threadIdx.x & 7;
  const unsigned ld = 16u * (unsigned)a.ldx, bytes = (unsigned)n * ld;
  const SynIn iQ = a.in[g][0], iS = a.in[g][1], iT = a.in[g][2];
  // rows of this order: row i at offset i ld; i = -1 wraps past the end
  const __amdgpu_buffer_rsrc_t rQ = brsrc(iQ.x1 + lms * 2 * a.ldx, bytes);
  const __amdgpu_buffer_rsrc_t rS = brsrc(VEC ? iS.x1 + lms * 2 * a.ldx : iQ.x1, VEC ? bytes : 0);
  const __amdgpu_buffer_rsrc_t rT = brsrc(VEC ? iT.x1 + lms * 2 * a.ldx : iQ.x1, VEC ? bytes : 0);
  const bool two = VEC && iT.mode == 2;
  const __amdgpu_buffer_rsrc_t rU = brsrc(two ? iT.x2 + lms * 2 * a.ldx : iQ.x1, two ? bytes : 0);
  const __amdgpu_buffer_rsrc_t rC = brsrc(VEC ? a.lcf + 4 * (lms + m) : iQ.x1, VEC ? 32u * (n + 1) : 0);
  unsigned oc[NS];  // offset of row r of the chunk
#pragma unroll
  for (int f = 0; f < NS; ++f) {
    const int b = bc0 + 8 * f + cc;
    oc[f] = b < a.B ? (unsigned)r * ld + 16u * (unsigned)b : kOut;
  }
  unsigned ol = 32u * (unsigned)r;
  const double sor2 = two && bc0 + cc < a.B ? a.or2[bc0 + cc] : 0.0;
  double dl = (double)(mo + r);  // degree of the item
  // raw inputs of the next chunk: Q (or the scalar tiles), S and T at l - 1, l,
  // l + 1, the second input of T, and the coupling coefficients
  double2 x0[NS], s3[3], t3[3], u3[3], cf;
  int ir = r;  // BIG: row of the item
  auto big = [&](const double* x, int i, int b) {
    return gld2(x + lms * 2 * a.ldx, i, n, 16L * a.ldx, b, a.B);
  };
  auto fetch = [&]() {
#pragma unroll
    for (int f = 0; f < NS; ++f) x0[f] = BIG ? big(iQ.x1, ir, bc0 + 8 * f + cc) : bld2(rQ, oc[f]);
    if constexpr (VEC) {
      cf = bld2(rC, ol);
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        if constexpr (BIG) {
          s3[q] = big(iS.x1, ir + q - 1, bc0 + cc);
          t3[q] = big(iT.x1, ir + q - 1, bc0 + cc);
          u3[q] = two ? big(iT.x2, ir + q - 1, bc0 + cc) : make_double2(0.0, 0.0);
        } else {
          const unsigned o = oc[0] + (unsigned)(q - 1) * ld;
          s3[q] = bld2(rS, o);
          t3[q] = bld2(rT, o);
          u3[q] = bld2(rU, o);  // zero without a second input
        }
      }
    }
  };
  const int row = (r & 1) * (CH / 2) + (r >> 1);  // parity-major rows
  // prefactor of a mode at degree l: k0 + k1 l(l+1)
  auto k0 = [](int mode) { return mode == 0 ? 1.0 : mode == 1 ? 0.0 : -1.0; };
  auto k1 = [](int mode) { return mode == 1 ? 1.0 : 0.0; };
  const double q0 = k0(iQ.mode), q1 = k1(iQ.mode), s0 = k0(iS.mode), s1 = k1(iS.mode);
  const double t0 = k0(iT.mode), t1 = k1(iT.mode);
  auto store = [&](int buf) {
    const double h = dl * (dl + 1.0);
    const double kq = q0 + q1 * h;
    double2 o[NF];
#pragma unroll
    for (int f = 0; f < NS; ++f) o[f] = cscale(x0[f], kq);
    if constexpr (VEC) {
      const double hq[3] = {h - 2.0 * dl, h, h + 2.0 * dl + 2.0};  // l(l+1) at l-1, l, l+1
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const double ks = s0 + s1 * hq[q], kt = t0 + t1 * hq[q], ku = sor2 * hq[q];
        s3[q] = cscale(s3[q], ks);
        t3[q] = make_double2(kt * t3[q].x + ku * u3[q].x, kt * t3[q].y + ku * u3[q].y);
      }
      o[1] = make_double2(cf.x * s3[0].x - cf.y * s3[2].x - dm * t3[1].y,
                          cf.x * s3[0].y - cf.y * s3[2].y + dm * t3[1].x);
      o[2] = make_double2(cf.y * t3[2].x - cf.x * t3[0].x - dm * s3[1].y,
                          cf.y * t3[2].y - cf.x * t3[0].y + dm * s3[1].x);
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) *reinterpret_cast<double2*>(&xs[buf][f][row][2 * cc]) = o[f];
  };
  auto advance = [&]() {  // to the next chunk's rows
#pragma unroll
    for (int f = 0; f < NS; ++f)
      if (oc[f] < kOut) oc[f] += (unsigned)CH * ld;
    ol += 32u * CH;
    ir += CH;
  };
  double4_t acc[NT][NF];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[i][f] = (double4_t){0, 0, 0, 0};
  // Table operands of one chunk, refilled in place.  Rows past the order's last
  // belong to the next order (or to the padding at the table's end) and meet
  // zero inputs; tiles past the last are computed on its operands and dropped.
  const double* tab = a.synP + a.mp_info[m * 8 + 4 * par + 1];
  unsigned tlo[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) tlo[i] = (unsigned)(kk * a.Hp + 16 * min(t0w + i, nt - 1) + col);
  double tc[SPC][NT];
  auto tload = [&](int s, int c0) {
    const double* base = tab + (long)((c0 >> 1) + 4 * s) * a.Hp;
#pragma unroll
    for (int i = 0; i < NT; ++i) tc[s][i] = base[tlo[i]];
  };
  fetch();
#pragma unroll
  for (int s = 0; s < SPC; ++s) tload(s, 0);
  store(0);
  __syncthreads();
  const int nch = (n1 + CH - 1) / CH;
  // MFMAs of chunk ch; LDS operands are read one step ahead, and the scheduling
  // barriers keep the compiler from reading the whole chunk's ahead (registers)
  auto compute = [&](int ch, auto more) {
    const double(*const x)[16] = xs[ch & 1][0] + par * (CH / 2) + kk;
    double xb[2][NF];
    auto xload = [&](int s) {
#pragma unroll
      for (int f = 0; f < NF; ++f) xb[s & 1][f] = x[f * CH + 4 * s][col];
    };
    xload(0);
#pragma unroll
    for (int s = 0; s < SPC; ++s) {
      if (s + 1 < SPC) xload(s + 1);
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[i][f] = mfma_f64(tc[s][i], xb[s & 1][f], acc[i][f]);
      if (more) tload(s, (ch + 1) * CH);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // every load of the loop is unconditional: a branch on the way would merge the
  // wait for the staged inputs with that for the table operands behind them
  for (int ch = 0; ch + 1 < nch; ++ch) {
    advance();
    fetch();
    compute(ch, std::true_type{});
    dl += (double)CH;
    store((ch & 1) ^ 1);  // last read before the previous barrier
    __syncthreads();
  }
  compute(nch - 1, std::false_type{});
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) smem[((w * NT + i) * 4 + v) * 64 + lane] = acc[i][f][v];
    __syncthreads();
    const int b = bc0 + (VEC ? 0 : 8 * f) + (col >> 1);
    double* F = a.F + fidx(VEC ? f * a.c_stride : 0, a.m_stride, a.Bout, 1, m, par, g * a.B + b) +
                (col & 1);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double other = smem[(((w ^ 1) * NT + i) * 4 + v) * 64 + lane];
        const int j = (t0w + i) * 16 + mfma_row(lane, v);
        if (j < a.H && b < a.B)
          F[4L * j * a.Bout] = par ? other - acc[i][f][v] : acc[i][f][v] + other;
      }
  }
}

int leg_synth_f64(int vector, const SynArgs& a, int n_m, hipStream_t st) {
  if (a.lcf == nullptr || a.l_max < 0) return MH_EINVAL;
  // an order's rows are addressed with 32-bit byte offsets below kOut, or else one by one
  const bool big = (long)(a.l_max + 64) * a.ldx * 16 >= (long)kOut;
  // theta tiles of 16 pairs over workgroups of two, four or six: the fewest
  // workgroups, since each stages the inputs anew (l_max = 383, 18 tiles: 2.59 ms
  // with six, 2.86 with four, 3.01 with two; l_max = 127, 6 tiles: 136, 159, 147 us)
  const int nt = mh_cdiv(a.H, 16), ny0 = mh_cdiv(nt, 6), NT = big ? 2 : mh_cdiv(mh_cdiv(nt, ny0), 2);
  const int ny = mh_cdiv(nt, 2 * NT);
  // scalar fields: three column tiles per workgroup where the batch has them and that
  // leaves enough workgroups for the 256 CUs, one tile otherwise (l_max = 341: 8 columns
  // in three tiles 42 us, in one 27; 17 columns 46 and 50)
  const long rows = (long)n_m * ny * a.ngroups;
  const bool three = vector || (!big && a.B > 16 && rows * mh_cdiv(a.B, 24) >= 1024);
  const long units =
      (long)a.ngroups * mh_cdiv(a.B, !vector && three ? 24 : 8) * ny * mh_cdiv(n_m, 8) * 8;
  if (units > 0x7fffffffL) return MH_EINVAL;
  const dim3 grid((unsigned)units), blk(256);
  if (big) {
    if (vector) hipLaunchKernelGGL((k_syn64<true, 3, 2, true>), grid, blk, 0, st, a, n_m);
    else hipLaunchKernelGGL((k_syn64<false, 1, 2, true>), grid, blk, 0, st, a, n_m);
    return mh_launch_status();
  }
#define MH_SYN64(NT)                                                                           \
  case NT:                                                                                     \
    if (vector) hipLaunchKernelGGL((k_syn64<true, 3, NT>), grid, blk, 0, st, a, n_m);          \
    else if (three) hipLaunchKernelGGL((k_syn64<false, 3, NT>), grid, blk, 0, st, a, n_m);     \
    else hipLaunchKernelGGL((k_syn64<false, 1, NT>), grid, blk, 0, st, a, n_m);                \
    break;
  switch (NT) {
    MH_SYN64(1) MH_SYN64(2) MH_SYN64(3)
    default: return MH_EINVAL;
  }
#undef MH_SYN64
  return mh_launch_status();
}

// ---------------------------------------------------------------- analysis
// One workgroup of four waves: order m, a window of degrees k0 .. (both
// parities, l = m + p + 2 k), and two fields of 8 complex columns that share
// every table operand: f_theta and f_phi of a pair (VEC), or 16 columns of a
// scalar component.  A wave takes 16 indices k, 15 after the one before it:
// the combination of neighbouring degrees needs one index of overlap between
// waves, so each wave works from its own accumulators and no sums are
// exchanged.  The hemisphere folds N + S and N - S of 32 theta pairs are staged
// in LDS (double-buffered); table operands stream through a ring of a whole
// chunk's steps, so that none waits behind the staged loads of that chunk.
template <bool VEC>
__global__ __launch_bounds__(256, 4) void k_ana64(AnaArgs a, int n_m) {
  __shared__ double fs[2][2][2][kChunk][16];  // [buffer][field][fold: +, -][pair][column]
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int CW = VEC ? 8 : 16;
  const int nbt = (a.B + CW - 1) / CW, gx = a.ncomp * nbt, tpx = a.ntiles / 8;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int* tl = a.tiles + 3 * (xcd * tpx + slot / gx);
  const int m = tl[0];
  if (m >= n_m) return;  // uniform per workgroup
  const int mo = m * (a.minc > 1 ? a.minc : 1);
  const int n = a.l_max + 1 - mo;
  // the windows of an order (consecutive in the list, this one number q of nw)
  // are walked window by window inside each column block, so that the Fourier
  // rows are read into the L2 once
  const int nw = tl[1] >> 16, q = tl[1] & 0xffff;
  const int lin = q * gx + slot % gx, cx = lin / nw;
  // the part of the window rotates over the waves (a wave stays on one SIMD, and
  // an order's last window has work for some of its parts only)
  const int kb = (lin - cx * nw) * kAnaWindow + 15 * ((w + cx) & 3);
  const bool active = kb == 0 || 2 * kb + 1 < n;  // some degree of this wave is <= l_max
  const int comp = cx / nbt, bc0 = (cx - comp * nbt) * CW;
  const int col = lane & 15, kk = lane >> 4;
  // staging: theta pair r of the chunk, complex column cc of both fields; the
  // rows of one component and order, zero past the last pair
  const int r = threadIdx.x >> 3, cc = threadIdx.x & 7;
  const unsigned ldb = 16u * (unsigned)a.Bin, bytes = 2u * (unsigned)a.H * ldb;
  const double* Fm = a.F + m * a.m_stride;
  const __amdgpu_buffer_rsrc_t rf[2] = {  // pairs: theta, phi
      brsrc(Fm + (VEC ? a.cf2[comp] : a.cf1[comp]) * a.c_stride, bytes),
      brsrc(Fm + a.cf1[comp] * a.c_stride, bytes)};
  unsigned of[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const int b = bc0 + (VEC ? 0 : 8 * f) + cc;
    of[f] = b < a.B ? 2u * r * ldb + 16u * (unsigned)b : kOut;
  }
  double2 rn[2], rs[2];
  auto fetch = [&]() {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      rn[f] = bld2(rf[f], of[f]);
      rs[f] = bld2(rf[f], of[f] + ldb);
      if (of[f] < kOut) of[f] += 2u * kChunk * ldb;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      *reinterpret_cast<double2*>(&fs[buf][f][0][r][2 * cc]) = cadd(rn[f], rs[f]);
      *reinterpret_cast<double2*>(&fs[buf][f][1][r][2 * cc]) = csub(rn[f], rs[f]);
    }
  };
  // table operands of this lane: index k of each tile and parity (k clamped to
  // the zero-padded row), theta pair 4 t + kk of step t
  constexpr int D = 8, SPC = kChunk / 4;
  const int* info = a.mp_info + m * 8;
  const int K16[2] = {info[3], info[7]};
  const double* tp[2] = {a.anaW + info[2], a.anaW + info[6]};
  unsigned to[2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
    to[p] = (unsigned)(kk * K16[p] + min(kb + col, K16[p] - 1));
  const int nsteps = (a.H + 3) / 4;  // the tables hold Hp >= roundup(H, 4) rows
  double4_t acc[2][2];  // [field][parity]
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int p = 0; p < 2; ++p) acc[f][p] = (double4_t){0, 0, 0, 0};
  double ring[D][2];
  auto tload = [&](double (&t)[2], int s) {
#pragma unroll
    for (int p = 0; p < 2; ++p) t[p] = (tp[p] + 4L * s * K16[p])[to[p]];
  };
  fetch();
#pragma unroll
  for (int d = 0; d < D; ++d) tload(ring[d], min(d, nsteps - 1));
  store(0);
  __syncthreads();
  const int nch = (a.H + kChunk - 1) / kChunk;
  // MFMAs of up to SPC steps of chunk ch (LDS operands read one step ahead)
  auto compute = [&](int ch, auto full) {
    const int buf = ch & 1;
    double xb[2][2][2];
    auto xload = [&](int s) {
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int p = 0; p < 2; ++p) xb[s & 1][f][p] = fs[buf][f][p][4 * s + kk][col];
    };
    xload(0);
#pragma unroll
    for (int s = 0; s < SPC; ++s) {
      const int t = ch * SPC + s;
      if (!full && t >= nsteps) break;
      if (s + 1 < SPC) xload(s + 1);
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int p = 0; p < 2; ++p) acc[f][p] = mfma_f64(ring[s % D][p], xb[s & 1][f][p], acc[f][p]);
      if (full) tload(ring[s % D], min(t + D, nsteps - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // as in the synthesis, waves without degrees run a loop of their own
  auto chunks = [&](auto act) {
    for (int ch = 0; ch + 1 < nch; ++ch) {
      fetch();
      if constexpr (decltype(act)::value) compute(ch, std::true_type{});
      store((ch & 1) ^ 1);  // last read before the previous barrier
      __syncthreads();
    }
    if constexpr (decltype(act)::value) compute(nch - 1, std::false_type{});
  };
  if (!active) {
    chunks(std::false_type{});
    return;
  }
  chunks(std::true_type{});
  const double dm = (double)mo;
  const long lms = a.lm_start[m];
  const double2* lcf = reinterpret_cast<const double2*>(a.lcf) + 2 * (lms + m);
  const int g = lane >> 4;  // accumulator row of element v: g + 4 v
#pragma unroll
  for (int p = 0; p < 2; ++p) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int kl = g + 4 * v, row = 2 * (kb + kl) + p;  // row = l - m
      // the last index of parity 1 and the first of parity 0 are the neighbouring
      // wave's, except at the start of the order
      const bool st = row < n && (p ? kl < 15 : (kl > 0 || kb == 0));
      if constexpr (!VEC) {
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          const int b = bc0 + 8 * f + (col >> 1);
          if (st && b < a.B) a.outS[comp][(lms + row) * 2L * a.ldo + 2 * b + (col & 1)] = acc[f][p][v];
        }
      } else {
        const double2 cl = lcf[2 * min(row, n) + 1];  // (l + 1) c_l, l c_{l+1}
        const double l = (double)(mo + row);
        const double inv = l > 0.0 ? 1.0 / (l * (l + 1.0)) : 0.0;
        const double Sv = ana_combine(acc[0][1 - p], acc[1][p][v], p, v, 1.0, cl, dm, lane);
        const double Tv = ana_combine(acc[1][1 - p], acc[0][p][v], p, v, -1.0, cl, dm, lane);
        const int b = bc0 + (col >> 1);
        if (st && b < a.B) {
          const long off = (lms + row) * 2L * a.ldo + 2 * b + (col & 1);
          a.outS[comp][off] = Sv * inv;
          if (a.outT[comp]) a.outT[comp][off] = Tv * inv;
        }
      }
    }
  }
}

// The same sums for few columns and low degrees, where a launch is as long as one
// wave's chain of MFMAs: one MFMA a step and wave instead of four.  A workgroup takes 8
// complex columns; a wave one parity, and one field of a window of 15 indices (VEC:
// the sums meet in LDS for the combination), or one of two such windows (scalar).  Every
// sum has the terms and the order of k_ana64's, so both give the same bits.  BIG as in
// k_syn64.
template <bool VEC, bool BIG = false>
__global__ __launch_bounds__(256, 4) void k_ana64s(AnaArgs a, int n_m, int sub) {
  constexpr int NF = VEC ? 2 : 1, WIN = VEC ? 15 : 30;  // fields; degree indices per workgroup
  __shared__ double fs[2][NF][2][kChunk][16];            // [buffer][field][fold: +, -][pair][column]
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nbt = (a.B + 7) / 8, gx = a.ncomp * nbt, tpx = a.ntiles / 8;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, gs = gx * sub;
  const int* tl = a.tiles + 3 * (xcd * tpx + slot / gs);
  const int m = tl[0];
  if (m >= n_m) return;  // uniform per workgroup
  const int mo = m * (a.minc > 1 ? a.minc : 1);
  const int n = a.l_max + 1 - mo;
  // windows inside each column block, as in k_ana64
  const int nw = (tl[1] >> 16) * sub, q = tl[1] & 0xffff;
  const int lin = q * gs + slot % gs, cx = lin / nw;
  const int k0 = (lin - cx * nw) * WIN;
  if (k0 > 0 && 2 * k0 + 1 >= n) return;  // uniform per workgroup: no degree <= l_max
  const int p = w & 1, f = VEC ? w >> 1 : 0;
  const int kb = VEC ? k0 : k0 + 15 * (w >> 1);
  const bool active = kb == 0 || 2 * kb + 1 < n;
  const int comp = cx / nbt, bc0 = (cx - comp * nbt) * 8;
  const int col = lane & 15, kk = lane >> 4;
  const int r = threadIdx.x >> 3, cc = threadIdx.x & 7;
  const unsigned ldb = 16u * (unsigned)a.Bin, bytes = 2u * (unsigned)a.H * ldb;
  const double* Fm = a.F + m * a.m_stride;
  const __amdgpu_buffer_rsrc_t rf[2] = {
      brsrc(Fm + (VEC ? a.cf2[comp] : a.cf1[comp]) * a.c_stride, bytes),
      brsrc(Fm + a.cf1[comp] * a.c_stride, bytes)};
  unsigned of = bc0 + cc < a.B ? 2u * r * ldb + 16u * (unsigned)(bc0 + cc) : kOut;
  double2 rn[NF], rs[NF];
  int ir = 2 * r;  // BIG: northern row of the pair
  auto fetch = [&]() {
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      if constexpr (BIG) {
        const double* Fc = Fm + (VEC && i == 0 ? a.cf2[comp] : a.cf1[comp]) * a.c_stride;
        rn[i] = gld2(Fc, ir, 2 * a.H, 16L * a.Bin, bc0 + cc, a.B);
        rs[i] = gld2(Fc, ir + 1, 2 * a.H, 16L * a.Bin, bc0 + cc, a.B);
      } else {
        rn[i] = bld2(rf[i], of);
        rs[i] = bld2(rf[i], of + ldb);
      }
    }
    if (of < kOut) of += 2u * kChunk * ldb;
    ir += 2 * kChunk;
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      *reinterpret_cast<double2*>(&fs[buf][i][0][r][2 * cc]) = cadd(rn[i], rs[i]);
      *reinterpret_cast<double2*>(&fs[buf][i][1][r][2 * cc]) = csub(rn[i], rs[i]);
    }
  };
  constexpr int D = 8, SPC = kChunk / 4;
  const int K16 = a.mp_info[m * 8 + 4 * p + 3];
  const double* tp = a.anaW + a.mp_info[m * 8 + 4 * p + 2];
  const unsigned to = (unsigned)(kk * K16 + min(kb + col, K16 - 1));
  const int nsteps = (a.H + 3) / 4;
  double4_t acc = (double4_t){0, 0, 0, 0};
  double ring[D];
  auto tload = [&](int s) { return (tp + 4L * s * K16)[to]; };
  fetch();
#pragma unroll
  for (int d = 0; d < D; ++d) ring[d] = tload(min(d, nsteps - 1));
  store(0);
  __syncthreads();
  const int nch = (a.H + kChunk - 1) / kChunk;
  auto compute = [&](int ch, auto full) {
    const double(*const x)[16] = fs[ch & 1][f][p] + kk;
    double xb[2];
    xb[0] = x[0][col];
#pragma unroll
    for (int s = 0; s < SPC; ++s) {
      const int t = ch * SPC + s;
      if (!full && t >= nsteps) break;
      if (s + 1 < SPC) xb[(s + 1) & 1] = x[4 * (s + 1)][col];
      acc = mfma_f64(ring[s % D], xb[s & 1], acc);
      if (full) ring[s % D] = tload(min(t + D, nsteps - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int ch = 0; ch + 1 < nch; ++ch) {
    fetch();
    if (active) compute(ch, std::true_type{});  // uniform per wave
    store((ch & 1) ^ 1);                        // last read before the previous barrier
    __syncthreads();
  }
  if (active) compute(nch - 1, std::false_type{});
  const int g = lane >> 4;
  const long lms = a.lm_start[m];
  const int b = bc0 + (col >> 1);
  if constexpr (!VEC) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int kl = g + 4 * v, row = 2 * (kb + kl) + p;
      const bool st = active && row < n && (p ? kl < 15 : (kl > 0 || kb == 0));
      if (st && b < a.B) a.outS[comp][(lms + row) * 2L * a.ldo + 2 * b + (col & 1)] = acc[v];
    }
  } else {
    // (every wave is active)  The buffer that the last chunk did not use: last read
    // before the previous barrier
    double(*const ex)[4][64] = reinterpret_cast<double(*)[4][64]>(&fs[nch & 1][0][0][0][0]);
    static_assert(sizeof(fs) / 2 >= 16 * 64 * sizeof(double), "exchange of the sums");
#pragma unroll
    for (int v = 0; v < 4; ++v) ex[w][v][lane] = acc[v];
    __syncthreads();
    double* out = f == 0 ? a.outS[comp] : a.outT[comp];
    double4_t opp, same;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      opp[v] = ex[2 * f + 1 - p][v][lane];
      same[v] = ex[2 * (1 - f) + p][v][lane];
    }
    const double2* lcf = reinterpret_cast<const double2*>(a.lcf) + 2 * (lms + m);
    const double sgn = f == 0 ? 1.0 : -1.0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int kl = g + 4 * v, row = 2 * (kb + kl) + p;
      const bool st = row < n && (p ? kl < 15 : (kl > 0 || kb == 0));
      const double l = (double)(mo + row);
      const double inv = l > 0.0 ? 1.0 / (l * (l + 1.0)) : 0.0;
      const double x = ana_combine(opp, same[v], p, v, sgn, lcf[2 * min(row, n) + 1], (double)mo, lane);
      if (st && b < a.B && out) out[(lms + row) * 2L * a.ldo + 2 * b + (col & 1)] = x * inv;
    }
  }
}

int leg_analysis_f64(int vector, const AnaArgs& a, hipStream_t st) {
  if (a.lcf == nullptr || a.l_max < 0) return MH_EINVAL;
  // the rows of an order past the reach of 32-bit byte offsets (as in leg_synth_f64)
  const bool big = (long)(a.H + kChunk) * 2 * a.Bin * 16 >= (long)kOut;
  // workgroups of k_ana64s per list entry: windows of 15 or 30 of its 60 indices (the
  // ones at k > 0 have degrees where 2 k + 1 <= l_max)
  const int win = vector ? 15 : 30, sub = std::min(kAnaWindow / win, 1 + std::max(0, a.l_max - 1) / (2 * win));
  // k_ana64s where its one MFMA a step and wave ends sooner: one window an order (three
  // quarters or half of k_ana64's waves have no degree there), few workgroups, and scalar
  // batches whose last tile of 16 columns is less than half full, as long as that is much
  // of the batch and the orders are short.  k_ana64 -> k_ana64s, us: scalar l_max = 16, 33
  // columns 4.4 -> 3.5; 60, 97: 8.3 -> 6.4; at the line 96, 64 (388 workgroups): 10.5 -> 10.3, 97
  // (679): 14.0 -> 14.8; part tiles 333, 8: 34 -> 29; 192, 33: 26 -> 24 and 216, 33: 31 -> 33; 267, 24:
  // 36 -> 32 and 383, 24: 80 -> 89.  Vector 16, 33: 5.7 -> 4.6; 60, 64 (488): 10.5 -> 8.8; three
  // pairs of 62 (1464): 18.6 -> 20.9; 96, 8 (97): 9.3 -> 7.4, 17 (291): 11.6 -> 11.9.
  const long wgs = (long)a.ncomp * mh_cdiv(a.B, vector ? 8 : 16) * a.ntiles;
  const bool small = big || sub == 1 || (vector ? wgs < (sub < 4 ? 512 : 192)
                                         : wgs < 400 || ((a.B - 1) % 16 < 8 && a.B * (long)a.l_max <= 6400));
  if (small) {
    const dim3 grid((unsigned)(a.ncomp * mh_cdiv(a.B, 8) * a.ntiles * sub)), blk(256);
    if (big && vector) hipLaunchKernelGGL((k_ana64s<true, true>), grid, blk, 0, st, a, a.n_m, sub);
    else if (big) hipLaunchKernelGGL((k_ana64s<false, true>), grid, blk, 0, st, a, a.n_m, sub);
    else if (vector) hipLaunchKernelGGL((k_ana64s<true>), grid, blk, 0, st, a, a.n_m, sub);
    else hipLaunchKernelGGL((k_ana64s<false>), grid, blk, 0, st, a, a.n_m, sub);
    return mh_launch_status();
  }
  const dim3 grid((unsigned)(a.ncomp * mh_cdiv(a.B, vector ? 8 : 16) * a.ntiles)), blk(256);
  if (vector) hipLaunchKernelGGL((k_ana64<true>), grid, blk, 0, st, a, a.n_m);
  else hipLaunchKernelGGL((k_ana64<false>), grid, blk, 0, st, a, a.n_m);
  return mh_launch_status();
}
