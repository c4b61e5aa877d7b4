// Blocked form of the truncated column-pivoted QR of the sparsify phase
// (gfx950): the greedy pivots of dgeqp3, found many at a time.
//
// C is k x N and wide (N is 5 to 40 times k at 64^3), and a pivot step over
// all of it is a chain of a device-wide argmax, a column broadcast and two
// passes: 12-15 us a step on the upper levels when the columns of a problem
// are spread over 8-32 workgroups that meet at every step (qp3.hip), with the
// columns of 500-1000 workgroups resident per launch.  Column norms never
// grow, so the pivots need not be looked for among all columns: of the 64
// columns with the largest norms, the best one is the best of all as long as
// its norm stays above the 65th norm (on ties, as long as its position is
// below every outsider's).  A round therefore is
//   panel   one workgroup per problem takes the 64 leading columns and
//           runs pivot steps on them alone until the best of them falls
//           under that bound (or 32 pivots, or the rank test ends it);
//   update  all columns <- (I - V T^T V^T) C for the round's reflectors on
//           the matrix cores, reading and writing C once, with the exact norms
//           of what is left.
// The pivots are those of the column-by-column algorithm: same largest norm,
// same first position on ties (LAPACK's swaps are kept as permutations), same
// stop at the first step i >= 1 with !(|r_ii| / |r_00| >= tol).  On the 64^3
// matrices a round finds 20-25 pivots of the 32 it may, so that one problem's
// step costs 1.4-2.2 us of its panel instead, and a batch needs neither
// co-residency nor barriers between workgroups.  All RRQRs of a factorization:
//   64^3 FP64 310 -> 74 ms (35 of them the update), 45^3 FP32 storage 84 -> 30,
//   33^3 FP64 31 -> 14.5, 15^3 5.3 -> 2.4, 2-D 128^2 4.2 -> 2.4
//
// Arithmetic is FP64 for both storage types.
#include <limits.h>

#include <algorithm>

#include "kcommon.hpp"
#include "descs.hpp"
#include "launch.hpp"

namespace spq {

constexpr double kDead = -2.0;  // norm slot of a pivoted column

__device__ __forceinline__ double wave_max(double v) {
  v = fmax(v, lane_xor<32>(v));
  v = fmax(v, lane_xor<16>(v));
  v = fmax(v, lane_xor<8>(v));
  v = fmax(v, lane_xor<4>(v));
  v = fmax(v, lane_xor<2>(v));
  return fmax(v, lane_xor<1>(v));
}
// wave-wide max / min of an int by DPP (every lane ends with the result)
template <bool MAX>
__device__ __forceinline__ int wave_ext(int v) {
  auto f = [](int a, int b) { return MAX ? max(a, b) : min(a, b); };
  v = f(v, lane_xor<1>(v));
  v = f(v, lane_xor<2>(v));
  v = f(v, lane_xor<4>(v));
  v = f(v, lane_xor<8>(v));
  v = f(v, lane_xor<16>(v));
  return f(v, lane_xor<32>(v));
}
// The lanes of `in` holding the wave's largest v, where v >= 0 or a common
// negative flag: by the high words, which order like the values, and by the
// low words only where those tie.
__device__ __forceinline__ unsigned long long wave_top(double v, bool in) {
  const int h = in ? __double2hiint(v) : INT_MIN;
  const int hm = wave_ext<true>(h);
  unsigned long long at = __ballot(in && h == hm);
  if (__popcll(at) > 1) {
    const int lo = in && h == hm ? (int)(__double2loint(v) ^ 0x80000000) : INT_MIN;
    const int lm = wave_ext<true>(lo);  // all lanes take part
    at = __ballot(in && h == hm && lo == lm);
  }
  return at;
}

// ---------------------------------------------------------------------------
// Squared column norms and the identity permutation: 64 columns x 4 row groups per
// workgroup, one pass over C (HBM bound).
constexpr int kInitCols = 64, kInitGroups = 4;
template <typename T>
__global__ __launch_bounds__(kInitCols * kInitGroups) void k_rrqr_init(const RrqrDesc<T>* __restrict__ descs,
                                                                       const int* __restrict__ tstart, int nd) {
  __shared__ double red[kInitGroups][kInitCols];
  const int p = find_owner(tstart, nd, blockIdx.x);
  const RrqrDesc<T> d = descs[p];
  const int t = blockIdx.x - tstart[p], lane = threadIdx.x & (kInitCols - 1), grp = threadIdx.x / kInitCols;
  const int j = t * kInitCols + lane;
  double s = 0;
  if (j < d.N) {
    const T* __restrict__ c = d.Ct + j;
#pragma unroll 8
    for (int r = grp; r < d.k; r += kInitGroups) {
      const double v = (double)c[(int64_t)r * d.ldc];
      s = fma(v, v, s);
    }
  }
  red[grp][lane] = s;
  __syncthreads();
  if (grp == 0 && j < d.N) {
#pragma unroll
    for (int q = 1; q < kInitGroups; ++q) s += red[q][lane];
    d.vn[j] = (s == s) ? s : -1.0;
    d.ipos[j] = j;
    d.perm[j] = j;
  }
  if (t == 0 && threadIdx.x == 0) {
    const int kmin = min(d.k, d.N);
    *d.st = RrqrState{0, 0, 0, kmin > 0 ? 0 : 1, 0.0};
  }
}

// ---------------------------------------------------------------------------
// The panel.  Lane l of every wave holds candidate column l, wave w the rows
// i0 + w + NW q (q < RW) of all 64, in registers.  Per pivot step the pivot's
// lane passes its RW entries to the other lanes of its wave through LDS (no
// barrier; by v_readlane the same two passes took 50 clocks a row, a scalar
// operand's wait with one wave per SIMD), each wave leaves one partial sum per column
// in LDS, and after one barrier all waves finish the sums, the reflector
// scalars, the norm downdates and the next argmax redundantly.  Row s leaves
// the registers at step s (zeros stay), so no pass masks rows.
// What bounds it: the latency of that chain, not the FMAs.
constexpr int kBins = 512;       // norm bins of the candidate selection: 1/64 octave each,
constexpr int kBinShift = 15;    // the last one everything below max / 256 (of squares: 1/32, 65536)

template <typename T, int NW, int RW>
__global__ __launch_bounds__(NW * kWave) void k_rrqr_panel(const RrqrDesc<T>* __restrict__ descs) {
  constexpr int NT = NW * kWave;
  constexpr int QM = kRrqrPivots / NW < RW ? kRrqrPivots / NW : RW;  // q's a pivot row can have
  // up to 48 rows per lane the pivot's entries stay in registers between the
  // two passes; beyond, both passes read them from LDS
  constexpr bool KEEP = RW <= 48;
  constexpr int XR = KEEP ? RW : 1;
  // norms kept in registers during the selection: N <= 64 NW HV columns
  constexpr int HV = NW == 1 ? 32 : (NW == 2 ? 24 : 16);
  __shared__ double part[2][NW][kWave];
  __shared__ double rowv[2][kWave];
  __shared__ __align__(16) double Gs[kRrqrPivots][kRrqrPivots];  // column s: products of v_s with the earlier reflectors
  __shared__ double taus[kRrqrPivots];
  __shared__ __align__(16) double xsh[NW][RW];
  __shared__ __align__(16) int hist[kBins];
  __shared__ int cidx[kRrqrCols], pwin[kRrqrPivots];
  __shared__ double wv_[NW];
  __shared__ int wp_[NW], wc_[NW], ws_[NW], wt_[NW];
  __shared__ int s_cut, s_before;

  const RrqrDesc<T> d = descs[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int i = __builtin_amdgcn_readfirstlane(d.st->next);
  if (d.st->done) {
    if (tid == 0) d.st->b = 0;
    return;
  }
  const int k = d.k, N = d.N, kmin = min(k, N), rows = k - i;
  const gptr<double> vn = to_global(d.vn);
  const gptr<int> ipos = to_global(d.ipos);

  // ---- the 64 candidates.  Slot 0 is the best column of all; then whole
  // norm bins from the top while they fit, and as much of the first one that
  // does not (in column order).  (bound, bpos): the best key left out.
  // Wave w scans columns [j0, j1), 64 at a time; all loads go out at once.
  const int chunk = ((N + kWave - 1) / kWave + NW - 1) / NW * kWave;
  const int j0 = w * chunk, j1 = min(N, j0 + chunk);
  const bool held = chunk <= HV * kWave;
  double hv[HV];
  if (held) {
#pragma unroll
    for (int u = 0; u < HV; ++u) {
      const int j = j0 + u * kWave + lane;
      hv[u] = j < j1 ? vn[j] : kDead;
    }
  }
  auto scan = [&](auto&& f) {  // f(column, its squared norm), uniform trip count per wave
    if (held) {
#pragma unroll
      for (int u = 0; u < HV; ++u)
        if (j0 + u * kWave < j1) f(j0 + u * kWave + lane, hv[u]);
    } else {
#pragma unroll 2
      for (int jb = j0; jb < j1; jb += kWave) f(jb + lane, jb + lane < j1 ? vn[jb + lane] : kDead);
    }
  };
  if (tid < kRrqrPivots) taus[tid] = 0.0;
  for (int q = tid; q < kBins; q += NT) hist[q] = 0;
  for (int q = tid; q < kRrqrPivots * kRrqrPivots; q += NT) (&Gs[0][0])[q] = 0.0;
  if (tid < kRrqrPivots) pwin[tid] = i + tid < N ? to_global(d.perm)[i + tid] : -1;
  double bv = kDead;
  scan([&](int, double v) { bv = fmax(bv, v); });
  bv = wave_max(bv);
  if (NW > 1) {
    if (lane == 0) wv_[w] = bv;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NW; ++q) bv = fmax(bv, wv_[q]);
  }
  // its first position
  int bp = INT_MAX, bc = -1;
  scan([&](int j, double v) {
    if (v == bv) {
      const int pj = ipos[j];
      if (pj < bp) { bp = pj; bc = j; }
    }
  });
  {
    const int pm = wave_ext<false>(bp);
    bc = __builtin_amdgcn_readlane(bc, __builtin_ctzll(__ballot(bp == pm)));
    bp = pm;
  }
  if (lane == 0) { wp_[w] = bp; wc_[w] = bc; }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NW; ++q)
    if (wp_[q] < bp) { bp = wp_[q]; bc = wc_[q]; }
  const int best = bc;
  const int hmax = __double2hiint(bv);
  // bin of a column (kBins: not a live column, or the best)
  auto bin = [&](int j, double v) {
    int q = v > 0 ? (hmax - __double2hiint(v)) >> kBinShift : kBins - 1;
    q = min(q, kBins - 1);
    return ((int)(v > -1.5) & (int)(j != best)) ? q : kBins;
  };
  scan([&](int j, double v) {
    const int q = bin(j, v);
    if (q < kBins - 1) atomicAdd(&hist[q], 1);
  });
  __syncthreads();
  if (w == 0) {
    constexpr int PL = kBins / kWave;  // consecutive bins per lane
    int h[PL];
#pragma unroll
    for (int q = 0; q < PL; ++q) h[q] = hist[lane * PL + q];
    int sum = 0;
#pragma unroll
    for (int q = 0; q < PL; ++q) sum += h[q];
    int inc = sum;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int u = __shfl_up(inc, o, kWave);
      if (lane >= o) inc += u;
    }
    const unsigned long long over = __ballot(inc > kRrqrCols - 1);
    if (over == 0) {
      if (lane == kWave - 1) { s_cut = kBins - 1; s_before = inc; }
    } else if (lane == __builtin_ctzll(over)) {
      int c = inc - sum, cutq = 0, cutc = c;
      bool open = true;
#pragma unroll
      for (int q = 0; q < PL; ++q) {
        const bool here = open & (c + h[q] > kRrqrCols - 1);
        cutq = here ? q : cutq;
        cutc = here ? c : cutc;
        open &= !here;
        c += h[q];
      }
      s_cut = lane * PL + cutq;
      s_before = cutc;
    }
  }
  __syncthreads();
  const int cut = s_cut, before = s_before;
  int ns = 0, nt = 0;
  scan([&](int j, double v) {
    const int q = bin(j, v);
    ns += __popcll(__ballot(q < cut));
    nt += __popcll(__ballot(q == cut));
  });
  if (lane == 0) { ws_[w] = ns; wt_[w] = nt; }
  __syncthreads();
  int so = 1, to = 1 + before, ties = 0;
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    if (q < w) { so += ws_[q]; to += wt_[q]; }
    ties += wt_[q];
  }
  const int nc = min(kRrqrCols, 1 + before + ties);
  if (tid == 0) cidx[0] = best;
  double bound = -3.0;
  const unsigned long long below = (1ull << lane) - 1;
  const int tie0 = to;
  scan([&](int j, double v) {
    const int q = bin(j, v);
    const unsigned long long ms = __ballot(q < cut), mt = __ballot(q == cut);
    const int slot = q < cut ? so + __popcll(ms & below) : (q == cut ? to + __popcll(mt & below) : INT_MAX);
    if (slot < kRrqrCols) cidx[slot] = j;
    bound = ((int)(q == cut) & (int)(slot >= kRrqrCols)) ? fmax(bound, v) : bound;
    so += __popcll(ms);
    to += __popcll(mt);
  });
  bound = wave_max(bound);
  __syncthreads();  // cidx is complete, wv_ / wp_ are read
  if (lane == 0) wv_[w] = bound;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NW; ++q) bound = fmax(bound, wv_[q]);
  int bpos = INT_MAX;  // the first position of those left out with that norm
  if (bound > -1.5) {
    int t = tie0;
    scan([&](int j, double v) {
      const bool tie = bin(j, v) == cut;
      const unsigned long long mt = __ballot(tie);
      if ((int)tie & (int)(v == bound) & (int)(t + __popcll(mt & below) >= kRrqrCols)) bpos = min(bpos, ipos[j]);
      t += __popcll(mt);
    });
    bpos = wave_ext<false>(bpos);
    if (NW > 1) {
      if (lane == 0) wp_[w] = bpos;
      __syncthreads();
#pragma unroll
      for (int q = 0; q < NW; ++q) bpos = min(bpos, wp_[q]);
    }
  }

  // ---- load the candidates
  const bool cand = lane < nc;
  const int jc = cand ? cidx[lane] : 0;
  double c[RW];
  {
    // row by row: a uniform row address plus the lane's column offset
    const T* src = d.Ct + (int64_t)min(i + w, k - 1) * d.ldc;
    const unsigned off = (unsigned)jc * (unsigned)sizeof(T);
    const int64_t step = (int64_t)NW * d.ldc;
#pragma unroll
    for (int q = 0; q < RW; ++q) {
      const double x = (double)load_at(src, off);
      c[q] = (cand && q * NW + w < rows) ? x : 0.0;
      if ((q + 1) * NW + w < rows) src += step;
    }
  }
  bool alive = cand;
  double v1 = cand ? vn[jc] : kDead, v2 = v1;  // squared norm: current, and at its last exact sum
  int pos = cand ? ipos[jc] : INT_MAX;
  int mine = -1;      // pivot number of this lane's column
  double vscale = 0;  // its reflector is c * vscale below row `mine`
  double r00 = d.st->r00, sure = d.tol * r00 * (1 + 1e-12);  // above `sure` the rank test needs no division
  bool stop = false;
  const double tol3z = sqrt(ldexp(1.0, -53));
  // f(q, x_q) for every row, the entries read 8 at a time one group ahead
  // (groups past the last row are skipped)
  auto pass = [&](auto&& f) {
    constexpr int CH = 8;
    double xb[2][CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) xb[0][u] = xsh[w][u];
#pragma unroll
    for (int q0 = 0; q0 < RW; q0 += CH) {
      if (q0 * NW + w < rows) {
        const int cur = (q0 / CH) & 1;
        if (q0 + CH < RW) {
#pragma unroll
          for (int u = 0; u < CH; ++u) xb[cur ^ 1][u] = xsh[w][q0 + CH + u];
        }
#pragma unroll
        for (int u = 0; u < CH; ++u) f(q0 + u, xb[cur][u]);
      }
    }
  };
  int s = 0;
  for (; s < kRrqrPivots && i + s < kmin; ++s) {
    // ---- the pivot: largest norm, first position
    unsigned long long at = wave_top(v1, alive);
    if (at == 0) break;  // no candidate left
    if (__popcll(at) > 1) {
      const bool t = (at >> lane) & 1;
      const int pm = wave_ext<false>(t ? pos : INT_MAX);
      at = __ballot(t && pos == pm);
    }
    const int p = __builtin_amdgcn_readfirstlane(__builtin_ctzll(at));
    const int ppos = __builtin_amdgcn_readlane(pos, p);
    const double top = lane_bcast(v1, p);
    if (s > 0 && !(top > bound || (top == bound && ppos < bpos))) break;  // an outsider may be the best
    // ---- row s of this lane's column leaves the registers
    double ci = 0;
    if (w == s % NW) {
      const int sq = s / NW;
#pragma unroll
      for (int g = 0; g < (QM + 3) / 4; ++g)
        if (sq / 4 == g) {
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (4 * g + u < QM && (sq & 3) == u) {
              ci = c[4 * g + u];
              c[4 * g + u] = 0.0;
            }
        }
    }
    // ---- x = the pivot column below row s; d = x . c for every candidate c
    if (lane == p) {
#pragma unroll
      for (int q = 0; q < RW; ++q) xsh[w][q] = c[q];
    }
    wave_sync();
    double a[4] = {0, 0, 0, 0};
    double x[XR];
    if (KEEP) {
#pragma unroll
      for (int q = 0; q < XR; ++q) x[q] = xsh[w][q];
#pragma unroll
      for (int q = 0; q < XR; ++q) a[q & 3] = fma(x[q], c[q], a[q & 3]);
    } else {
      pass([&](int q, double v) { a[q & 3] = fma(v, c[q], a[q & 3]); });
    }
    double dot = (a[0] + a[1]) + (a[2] + a[3]);
    const int buf = s & 1;
    if (NW > 1) {
      part[buf][w][lane] = dot;
      if (w == s % NW) rowv[buf][lane] = ci;
      __syncthreads();
      dot = part[buf][0][lane];
#pragma unroll
      for (int q = 1; q < NW; ++q) dot += part[buf][q][lane];
      ci = rowv[buf][lane];
    }
    // row s of the reflectors so far
    if (w == 0 && mine >= 0)
      store_at(d.V + (int64_t)(i + s) * d.ldv + i, (unsigned)mine * (unsigned)sizeof(T), (T)(ci * vscale));
    // ---- reflector u = (head; x), H = I - g u u^T, g = tau / head^2 = -1 / (beta
    // head): one reciprocal square root and one reciprocal (Newton-refined)
    // serve beta, g, tau = -head / beta and scal = 1 / head.  Where the
    // squares leave the range the scaled forms take over.
    const double ssq = lane_bcast(dot, p), alpha = lane_bcast(ci, p);
    double beta = alpha, head = 0, tau = 0, scal = 0, f = 0;
    const bool upd = (int)alive & (int)(lane != p);
    const double n2 = fma(alpha, alpha, ssq);
    if (ssq > 0 && n2 > 1e-280 && n2 < 1e280) {
      beta = -copysign(sqrt_nr(n2), alpha);
      head = alpha - beta;
      const double r = rcp_nr(beta * head);
      f = fma(head, ci, dot) * -r;
      scal = beta * r;
      tau = -(head * head) * r;
    } else if (ssq > 0) {
      beta = -copysign(hypot(alpha, sqrt(ssq)), alpha);
      head = alpha - beta;
      scal = 1.0 / head;
      tau = (beta - alpha) / beta;
      f = tau * scal * fma(scal, dot, ci);
    }
    if (i + s == 0) {
      r00 = fabs(beta);
      sure = d.tol * r00 * (1 + 1e-12);
    } else if (!(fabs(beta) > sure) && !(fabs(beta) / r00 >= d.tol)) {
      stop = true;
      break;
    }
    // ---- c -= f u
    f = upd ? f : 0.0;
    if (KEEP) {
#pragma unroll
      for (int q = 0; q < XR; ++q) c[q] = fma(-f, x[q], c[q]);
    } else {
      pass([&](int q, double v) { c[q] = fma(-f, v, c[q]); });
    }
    if (w == 0) {
      if (mine >= 0) Gs[mine][s] = vscale * fma(scal, dot, ci);  // v_mine . v_s
      else if (lane == p) store_at(d.V + (int64_t)(i + s) * d.ldv + i, (unsigned)s * (unsigned)sizeof(T), T(1));
    }
    // ---- norm downdate: that of dlaqp2 on squares, |c|^2 - c_s^2, with a
    // fresh sum where it has cancelled to sqrt(eps) of the last one
    bool need = false;
    if (upd && v1 > 0.0) {
      const double cs = fma(-f, head, ci);
      v1 = fma(-cs, cs, v1);
      v1 = v1 < 0.0 ? 0.0 : v1;
      need = v1 <= tol3z * v2;
    }
    if (__ballot(need) != 0) {
      double e = 0;
      if (i + s < k - 1) {
#pragma unroll
        for (int q = 0; q < RW; ++q) e = fma(c[q], c[q], e);
        if (NW > 1) {
          __syncthreads();  // this step's partials are read
          part[buf][w][lane] = e;
          __syncthreads();
          e = part[buf][0][lane];
#pragma unroll
          for (int q = 1; q < NW; ++q) e += part[buf][q][lane];
        }
      }
      if (need) {
        v1 = e;
        v2 = e;
      }
    }
    if (upd && !(v1 == v1)) v1 = -1.0;
    if (lane == p) {
      mine = s;
      vscale = scal;
      alive = false;
    }
    if (alive && pos == i + s) pos = ppos;
    if (w == NW - 1 && lane == p) {  // wave 0 has the V row and the products
      taus[s] = tau;
      to_global_mut(d.tau)[i + s] = (T)tau;
      // LAPACK swap of positions i + s and ppos
      const int qcol = pwin[s];
      to_global_mut(d.perm)[ppos] = qcol;
      to_global_mut(d.ipos)[qcol] = ppos;
      to_global_mut(d.perm)[i + s] = jc;
      to_global_mut(d.ipos)[jc] = i + s;
      if (ppos - i < kRrqrPivots) pwin[ppos - i] = qcol;
    }
  }
  const int b = s;
  if (tid == 0) *d.st = RrqrState{i, b, i + b, stop || i + b >= kmin ? 1 : 0, r00};
  if (b == 0) return;
  // ---- the rest of the round's reflectors: columns [i, i + 32) of V, by rows,
  // zero above the diagonal, where there is no pivot and in the rows up to
  // the next 16 (a row that left the registers was stored up to its diagonal
  // then; the pivot columns of C itself are left to the update)
  {
    const unsigned long long taken = __ballot(mine >= 0);
    const int slot = mine >= 0 ? mine : b + __popcll(~taken & below);
    const int rows16 = (rows + 15) / 16 * 16, left = b + (stop ? 1 : 0);
    if (slot < kRrqrPivots) {
      T* vd = d.V + (int64_t)(i + w) * d.ldv + i;
      const unsigned voff = (unsigned)slot * (unsigned)sizeof(T);
#pragma unroll
      for (int q = 0; q < RW; ++q) {
        const int r = q * NW + w;
        const bool reg = q >= QM || r >= left;
        const double v = reg ? c[q] * vscale : 0.0;  // vscale = 0 without a pivot
        if (r < rows16 && (reg || slot > r || (slot == r && r >= b))) store_at(vd, voff, (T)v);
        vd += (int64_t)NW * d.ldv;
      }
    }
  }
  // ---- T factor, by one wave: lane r forms row r.  T(r, l) = -tau_l acc_l is
  // final when its turn comes and is then added to all later columns, so
  // the sums never wait for one another.
  __syncthreads();
  if (w == NW - 1 && lane < kRrqrPivots) {
    const gmut<double> tm = to_global_mut(d.Tm) + lane * kRrqrPivots;
    double t[kRrqrPivots];
#pragma unroll
    for (int j = 0; j < kRrqrPivots; ++j) t[j] = 0.0;
#pragma unroll
    for (int l = 0; l < kRrqrPivots; ++l) {
      const double v = taus[l] * (lane == l ? 1.0 : -t[l]);
      tm[l] = v;
#pragma unroll
      for (int j = l + 1; j < kRrqrPivots; ++j) t[j] = fma(v, Gs[l][j], t[j]);
    }
  }
}

// ---------------------------------------------------------------------------
// The update, C <- C - V (T^T (V^T C)) on rows >= i0, and the squared norms of the
// rows below the round's pivots: 16 columns by 4 waves, the 16-row tiles of
// C dealt to the waves.  The FP64 matrix instruction leaves row l / 16 + 4 c of
// a result tile in accumulator c of lane l, which is also where it wants row
// l / 16 of the c-th 4-row slice of its right operand: C is loaded once, as
// the accumulators of C - V Z, and the same registers are the operand of
// V^T C.  The waves' V^T C are summed in LDS (21 KB, so that 7 workgroups share
// a CU: between load and store a workgroup waits for memory twice and at
// two barriers, and only other workgroups fill that).  A wave per 16 or 32
// columns, with all rows in registers and no LDS or barrier, held 1-2 waves
// per SIMD and was 1.7-2.6x slower.
//
// A column pivoted in this round becomes its column of R: the rows below its
// pivot row are stored as zeros.  Columns pivoted earlier are left alone.
constexpr int kUThreads = 256, kUCols = 16;
template <typename T, int RT>  // row tiles per wave
__global__ __launch_bounds__(kUThreads) void k_rrqr_update(const RrqrDesc<T>* __restrict__ descs,
                                                           const int* __restrict__ tstart, int nd) {
  using V4 = Mfma<double>::v4;
  constexpr int P = kRrqrPivots, NWV = kUThreads / kWave, LD = kUCols + 1;
  __shared__ double Ys[NWV][P][LD];
  __shared__ double Zs[P][LD];
  const int p = find_owner(tstart, nd, blockIdx.x);
  const RrqrDesc<T> d = descs[p];
  const RrqrState st = *d.st;
  if (st.b == 0) return;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), c16 = lane & 15, k4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int j = (blockIdx.x - tstart[p]) * kUCols + c16;
  const int rows = d.k - st.i0, b = st.b;
  const bool two = b > 16, in = j < d.N;
  const int64_t ldc = d.ldc, ldv = d.ldv;
  const gmut<T> C = to_global_mut(d.Ct) + j + (int64_t)st.i0 * ldc;
  const gptr<T> V = to_global((const T*)d.V) + (int64_t)st.i0 * ldv + st.i0;
  V4 c[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int rb = (t * NWV + w) * 16;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = rb + 4 * q + k4;
      c[t][q] = (r < rows && in) ? (double)C[(int64_t)r * ldc] : 0.0;
    }
  }
  // position of the column relative to this round's pivots (< 0: pivoted before)
  const int piv = in ? to_global((const int*)d.ipos)[j] - st.i0 : -1;
  V4 y0 = V4{0, 0, 0, 0}, y1 = V4{0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int rb = (t * NWV + w) * 16;
    if (rb < rows) {
      const gptr<T> vr = V + (int64_t)(rb + k4) * ldv + c16;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        y0 = Mfma<double>::mac((double)vr[(int64_t)4 * q * ldv], c[t][q], y0);
        if (two) y1 = Mfma<double>::mac((double)vr[(int64_t)4 * q * ldv + 16], c[t][q], y1);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    Ys[w][4 * q + k4][c16] = y0[q];
    Ys[w][16 + 4 * q + k4][c16] = y1[q];
  }
  __syncthreads();
  // Z = -T^T Y (T upper triangular), 16 rows by each of two waves
  if (w < 2) {
    V4 z = V4{0, 0, 0, 0};
    if (w == 0 || two) {
#pragma unroll
      for (int kk = 0; kk < P / 4; ++kk) {
        if (kk < 4 || w == 1) {
          const int l = 4 * kk + k4;
          double ys = Ys[0][l][c16];
#pragma unroll
          for (int q = 1; q < NWV; ++q) ys += Ys[q][l][c16];
          z = Mfma<double>::mac(to_global((const double*)d.Tm)[l * P + w * 16 + c16], ys, z);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) Zs[w * 16 + 4 * q + k4][c16] = piv >= 0 ? -z[q] : 0.0;
  }
  __syncthreads();
  const bool own = piv >= 0 && piv < b;  // pivoted in this round
  double nr = 0;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int rb = (t * NWV + w) * 16;
    if (rb < rows) {
      // the contraction runs over the reflectors in the order that lets a
      // lane read four of its row at once: k-slot k4 of step kk is reflector
      // 16 (kk / 4) + 4 k4 + kk % 4
      const gptr<T> vr = V + (int64_t)(rb + c16) * ldv + 4 * k4;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) c[t] = Mfma<double>::mac((double)vr[kk], Zs[4 * k4 + kk][c16], c[t]);
      if (two) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) c[t] = Mfma<double>::mac((double)vr[16 + kk], Zs[16 + 4 * k4 + kk][c16], c[t]);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = rb + 4 * q + k4;
        const T x = (own && r > piv) ? T(0) : (T)c[t][q];
        // after the last round only R's rows are read again
        if (r < rows && (r < b || !st.done) && piv >= 0) C[(int64_t)r * ldc] = x;
        if (r >= b) nr = fma((double)x, (double)x, nr);  // rows beyond the last are zero
      }
    }
  }
  if (st.done) return;
  nr += lane_xor<16>(nr);
  nr += lane_xor<32>(nr);
  // the Y sums are read (second barrier): their first rows take the norms
  if (k4 == 0) Ys[w][0][c16] = nr;
  __syncthreads();
  if (w == 0 && k4 == 0 && piv >= 0) {
#pragma unroll
    for (int q = 1; q < NWV; ++q) nr += Ys[q][0][c16];
    to_global_mut(d.vn)[j] = own ? kDead : (nr == nr ? nr : -1.0);
  }
}

// ---------------------------------------------------------------------------
namespace {
struct Form { int nw, rw; };
// (waves, rows per lane), each holding nw * rw rows; a launch takes the least
// that holds its rows.  Up to 48 rows four waves are the quickest for one
// problem (the selection's scans are split as well), but their redundant
// scalar work crowds the SIMDs once there are more waves than two per SIMD:
// launches of more than kCrowd problems use one wave each, which needs no
// barrier (1024 problems of 42 rows: 78 us a round, 4 waves 120 us).
constexpr Form kForms[] = {{1, 16}, {1, 32}, {1, 48}, {4, 12}, {2, 32}, {4, 28}, {4, 40},
                           {8, 28}, {8, 36}, {8, 48}, {8, 64}, {8, 88}};
constexpr int kNumForms = sizeof(kForms) / sizeof(kForms[0]), kCrowd = 512;
}  // namespace
int rrqr_form(int k, int nd) {
  for (int f = nd > kCrowd ? 0 : 3; f < kNumForms; ++f)
    if (k <= kForms[f].nw * kForms[f].rw) return f + 1;
  return 0;
}
int rrqr_form_waves(int form) { return form >= 1 && form <= kNumForms ? kForms[form - 1].nw : 0; }
int rrqr_form_rows(int form) { return form >= 1 && form <= kNumForms ? kForms[form - 1].rw : 0; }
int rrqr_init_tiles(int N) { return std::max(1, (N + kInitCols - 1) / kInitCols); }

template <typename T>
void launch_rrqr_init(hipStream_t s, const RrqrDesc<T>* d, const int* tstart, int nd, int ntiles) {
  if (nd <= 0 || ntiles <= 0) return;
  hipLaunchKernelGGL((k_rrqr_init<T>), dim3(ntiles), dim3(kInitCols * kInitGroups), 0, s, d, tstart, nd);
}
template <typename T>
void launch_rrqr_panel(hipStream_t s, const RrqrDesc<T>* d, int nd, int form) {
  if (nd <= 0) return;
  auto go = [&](auto nw, auto rw) {
    constexpr int NW = decltype(nw)::value, RW = decltype(rw)::value;
    hipLaunchKernelGGL((k_rrqr_panel<T, NW, RW>), dim3(nd), dim3(NW * kWave), 0, s, d);
  };
#define SPQ_FORM(f)                                              \
  case f + 1:                                                    \
    go(std::integral_constant<int, kForms[f].nw>{}, std::integral_constant<int, kForms[f].rw>{}); \
    break;
  switch (form) {
    SPQ_FORM(0) SPQ_FORM(1) SPQ_FORM(2) SPQ_FORM(3) SPQ_FORM(4) SPQ_FORM(5) SPQ_FORM(6) SPQ_FORM(7) SPQ_FORM(8)
    SPQ_FORM(9) SPQ_FORM(10) SPQ_FORM(11)
  }
#undef SPQ_FORM
}
int rrqr_update_cols() { return kUCols; }
template <typename T>
void launch_rrqr_update(hipStream_t s, const RrqrDesc<T>* d, const int* tstart, int nd, int ntiles, int kmax) {
  if (nd <= 0 || ntiles <= 0) return;
  auto go = [&](auto rt) {
    hipLaunchKernelGGL((k_rrqr_update<T, decltype(rt)::value>), dim3(ntiles), dim3(kUThreads), 0, s, d, tstart, nd);
  };
  if (kmax <= 64) go(std::integral_constant<int, 1>{});
  else if (kmax <= 128) go(std::integral_constant<int, 2>{});
  else if (kmax <= 192) go(std::integral_constant<int, 3>{});
  else if (kmax <= 320) go(std::integral_constant<int, 5>{});
  else if (kmax <= 512) go(std::integral_constant<int, 8>{});
  else go(std::integral_constant<int, 11>{});
}
template void launch_rrqr_init<double>(hipStream_t, const RrqrDesc<double>*, const int*, int, int);
template void launch_rrqr_init<float>(hipStream_t, const RrqrDesc<float>*, const int*, int, int);
template void launch_rrqr_panel<double>(hipStream_t, const RrqrDesc<double>*, int, int);
template void launch_rrqr_panel<float>(hipStream_t, const RrqrDesc<float>*, int, int);
template void launch_rrqr_update<double>(hipStream_t, const RrqrDesc<double>*, const int*, int, int, int);
template void launch_rrqr_update<float>(hipStream_t, const RrqrDesc<float>*, const int*, int, int, int);

}  // namespace spq
