// Householder panel kernels (gfx950).
//
// k_panel_r: factors one NB-wide column block [jb, jb+w) of every panel in
// the batch: dlarfg-convention reflectors (beta = -sign(alpha) * ||x||,
// tau = (beta - alpha) / beta, v(0) = 1), the reflector applied to the
// remaining columns of the block, and the block's compact-WY factor T
// (forward, columnwise: T(0:j,j) = -tau_j T(0:j,0:j) V^T v_j).  The caller
// applies the block to the trailing columns (k_larfb).
#include "kcommon.hpp"
#include "descs.hpp"
#include "launch.hpp"

namespace spq {

constexpr int kNB = 32;
constexpr int kThreads = 256;

// The 32 x 32 T factor (ld 32) of reflectors with pairwise products
// Gs[l][j] = v_l . v_j (l < j) and scalars taus (zero past the last one), by the
// first 32 lanes of one wave: lane r forms row r.  T(r, l) = -taus[l] acc_l is
// final when its turn comes and is then added to all later columns, so the
// sums never wait for one another.
template <typename T>
__device__ __forceinline__ void t_factor(const T (&Gs)[kNB][kNB], const T (&taus)[kNB], gmut<T> Tb) {
  const int lane = threadIdx.x & (kWave - 1);
  if (lane >= kNB) return;
  T t[kNB];
#pragma unroll
  for (int j = 0; j < kNB; ++j) t[j] = T(0);
#pragma unroll
  for (int l = 0; l < kNB; ++l) {
    const T v = lane > l ? T(0) : taus[l] * (lane == l ? T(1) : -t[l]);
    Tb[lane + l * kNB] = v;
#pragma unroll
    for (int j = l + 1; j < kNB; ++j) t[j] = fma(v, Gs[l][j], t[j]);
  }
}

// The panel step.  A wave holds 8 Q rows of the block's 32 columns in
// registers: lane (c8, g) = (lane / 8, lane % 8) the columns 4 c8 .. 4 c8 + 3 of
// the rows g, g + 8, ... of its 8-row groups, which are dealt to the NW waves
// in turn.  Column step j needs d_c = sum_{r > j} x_r A(r, c) for all 32
// columns (x = column j below the diagonal): the 8 lanes that hold column j pass
// it to the wave through LDS (no barrier; Q values a lane serve 4 Q FMAs), a sum
// is finished over 8 lanes by 4 exchanges, and over the waves through LDS
// behind the step's one barrier.  d_j is ||x||^2, and with row j (published by
// the wave that holds it)
//   v_j^T A(:, c) = A(j, c) + scal * d_c
// gives both the update of the later columns and the products with the
// earlier reflectors for T.  Row j is final after step j in every column: it
// is stored and its registers are zeroed, so no pass masks rows.  (A column that is
// not finite meets the earlier ones as x times zero, so that their V entries are
// not kept; the block's T is not finite then, nor anything it is applied to.)
// What bounds it: the latency of one step, and a launch has few panels (1-24
// per elimination wave above level 2), so a panel stays in one workgroup as
// long as its registers hold it (1280 rows in FP64).  One row per thread, 256
// rows per workgroup and workgroups that met at every step took 4.4 us a step
// at 64^3 (the 32-value reduction over 64 lanes alone 170 instructions); now
// 1.4 us (33^3).  All panels of a factorization: 64^3 104 -> 47 ms, 33^3 29 -> 9.6,
// 45^3 FP32 60 -> 15, 2-D 128^2 4.9 -> 2.1.
// Larger panels are split over workgroups of 512 rows that exchange their sums
// once per column, each value with its own arrival: a slot holds the value's
// complement and is zero until then, so a reader polls the values themselves
// (one trip through memory for the store and one for the load; a counter
// barrier between them takes three).  Every step has its own slots.
template <typename T>
__device__ __forceinline__ T panel_rcp(T v) {
  if constexpr (sizeof(T) == 8) return rcp_nr(v);
  else return T(1) / v;
}
template <typename T>
__device__ __forceinline__ T panel_sqrt(T v) {
  if constexpr (sizeof(T) == 8) return sqrt_nr(v);
  else return sqrt(v);
}
template <typename T, int NW, int Q>
__global__ __launch_bounds__(NW * kWave) void k_panel_r(const PanelDesc<T>* __restrict__ descs,
                                                        const int* __restrict__ wstart, int nd, int jb) {
  constexpr int QX = Q + 16 / (int)sizeof(T);  // padded: the 8 row groups of a read fall into different banks
  constexpr int QR = NW >= 4 ? 1 : 4 / NW;     // 8-row groups of a wave among the first 32 rows
  constexpr bool KEEP = 5 * Q * sizeof(T) <= 640;  // x stays in registers from the sums to the update
  __shared__ __align__(16) T xsh[NW][8][QX];
  __shared__ T part[2][NW][kNB], rowv[2][kNB], dsh[kNB];
  __shared__ __align__(16) T fsh[NW][kNB];
  __shared__ __align__(16) T Gs[kNB][kNB];
  __shared__ T taus[kNB], vsc[kNB];
  const int p = ((int)gridDim.x == nd) ? (int)blockIdx.x : find_owner(wstart, nd, blockIdx.x);
  const PanelDesc<T> d = descs[p];
  const int kk = min(d.m, d.k);
  if (jb >= kk) return;  // uniform over the problem's workgroups
  const int wg = blockIdx.x - wstart[p], nwg = d.nwg;
  const int w32 = min(kNB, kk - jb), ncb = min(kNB, d.k - jb);
  const int tid = threadIdx.x, lane = tid & (kWave - 1), g = lane & 7, c8 = lane >> 3, lc = lane & (kNB - 1);
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int64_t ld = d.ld;
  const int r0 = jb + wg * (8 * Q * NW);  // this workgroup's first row
  const int rows = d.m - r0;
  // row 8 (q NW + w) + g of the workgroup, column 4 c8 + t
  T a[Q][4];
  {
    const gptr<T> src = to_global((const T*)d.P) + (int64_t)r0 + 8 * w + g + (int64_t)(jb + 4 * c8) * ld;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int r = 8 * (q * NW + w) + g;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        a[q][t] = ((int)(r < rows) & (int)(4 * c8 + t < ncb)) ? src[8 * q * NW + (int64_t)t * ld] : T(0);
    }
  }
  for (int q = tid; q < kNB * kNB; q += NW * kWave) (&Gs[0][0])[q] = T(0);
  if (tid < kNB) taus[tid] = T(0);
  T vscale = T(0);  // of column lc: its reflector is the register value times vscale
  for (int jj = 0; jj < w32; ++jj) {
    const int buf = jj & 1, gr = jj & 7, tp = jj & 3, cp = jj >> 2;
    // ---- row j leaves the registers
    if (wg == 0 && w == (jj >> 3) % NW) {
      const int qr = (jj >> 3) / NW;
#pragma unroll
      for (int q = 0; q < QR; ++q)
        if (q == qr) {
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            if (g == gr) rowv[buf][4 * c8 + t] = a[q][t];
            a[q][t] = g == gr ? T(0) : a[q][t];
          }
        }
    }
    // ---- x, and this wave's part of the sums
    if (c8 == cp) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (t == tp) {
#pragma unroll
          for (int q = 0; q < Q; ++q) xsh[w][g][q] = a[q][t];
        }
    }
    wave_sync();
    T x[KEEP ? Q : 1];
    if (KEEP) {
#pragma unroll
      for (int q = 0; q < Q; ++q) x[KEEP ? q : 0] = xsh[w][g][q];
    }
    T s[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const T xq = KEEP ? x[KEEP ? q : 0] : xsh[w][g][q];
#pragma unroll
      for (int t = 0; t < 4; ++t) s[t] = fma(xq, a[q][t], s[t]);
    }
    {
      // over the 8 lanes of a column group: two halving exchanges, then one
      // full one; lane g ends with column 4 c8 + 2 (g & 1) + (g >> 1 & 1)
      const bool b0 = g & 1, b1 = g & 2;
      T u0 = (b0 ? s[2] : s[0]) + lane_xor<1>(b0 ? s[0] : s[2]);
      T u1 = (b0 ? s[3] : s[1]) + lane_xor<1>(b0 ? s[1] : s[3]);
      T v = (b1 ? u1 : u0) + lane_xor<2>(b1 ? u0 : u1);
      v += lane_xor<4>(v);
      if (g < 4) part[buf][w][4 * c8 + 2 * (g & 1) + (g >> 1)] = v;
    }
    if (NW > 1) __syncthreads();
    else wave_sync();
    T dot = part[buf][0][lc];
#pragma unroll
    for (int q = 1; q < NW; ++q) dot += part[buf][q][lc];
    if (nwg > 1) {
      // wave 0 exchanges the sums (lanes < 32) and row j (lanes >= 32)
      if (w == 0) {
        slot_put(d.part, (int64_t)(jj * nwg + wg) * (2 * kNB) + lane, wg == 0 || lane < kNB,
                 lane < kNB ? dot : rowv[buf][lc]);
        // the sums of all workgroups in workgroup order; row j from the first
        const T v = slot_sum<T, 8>(d.part + (int64_t)jj * nwg * (2 * kNB) + lane, 2 * kNB, lane < kNB ? nwg : 1, nwg,
                                   d.err);
        if (lane < kNB) dsh[lane] = v;
        else if (wg != 0) rowv[buf][lc] = v;
      }
      __syncthreads();
      dot = dsh[lc];
    }
    const T ci = rowv[buf][lc];
    // ---- reflector scalars (alike in every thread and workgroup): u = (head; x),
    // H = I - u u^T / (-beta head); scaled forms where the squares leave the range
    const T ssq = lane_bcast(dot, jj), alpha = lane_bcast(ci, jj);
    T beta = alpha, head = T(0), tau = T(0), scal = T(0), f = T(0);
    const T n2 = fma(alpha, alpha, ssq);
    constexpr T lo = sizeof(T) == 8 ? T(1e-280) : T(1e-30), hi = sizeof(T) == 8 ? T(1e280) : T(1e30);
    if (ssq > T(0) && n2 > lo && n2 < hi) {
      beta = -copysign(panel_sqrt(n2), alpha);
      head = alpha - beta;
      const T r = panel_rcp(beta * head);
      f = fma(head, ci, dot) * -r;
      scal = beta * r;
      tau = -(head * head) * r;
    } else if (ssq > T(0)) {
      beta = -copysign(hypot(alpha, sqrt(ssq)), alpha);
      head = alpha - beta;
      scal = T(1) / head;
      tau = (beta - alpha) / beta;
      f = tau * scal * fma(scal, dot, ci);
    }
    const T vdot = vscale * fma(scal, dot, ci);  // v_lc . v_j for the earlier reflectors
    f = (lc > jj && lc < ncb) ? f : T(0);
    if (lane < kNB) fsh[w][lc] = f;
    wave_sync();
    // ---- a -= f x (column j and the earlier ones keep their x)
    {
      T ft[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) ft[t] = fsh[w][4 * c8 + t];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const T xq = KEEP ? x[KEEP ? q : 0] : xsh[w][g][q];
#pragma unroll
        for (int t = 0; t < 4; ++t) a[q][t] = fma(-ft[t], xq, a[q][t]);
      }
    }
    if (wg == 0 && w == NW - 1 && lane < ncb) {
      const T v = lc < jj ? ci * vscale : (lc == jj ? beta : fma(-f, head, ci));
      to_global_mut(d.P)[(int64_t)(jb + jj) + (int64_t)(jb + lc) * ld] = v;
      if (lc < jj) Gs[lc][jj] = vdot;
      if (lc == jj) {
        taus[jj] = tau;
        to_global_mut(d.tau)[jb + jj] = tau;
      }
    }
    if (lc == jj) vscale = scal;
  }
  if (w == 0 && lane < kNB) vsc[lc] = vscale;
  __syncthreads();
  // ---- the rows below the block's triangle
  {
    T vt[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) vt[t] = vsc[4 * c8 + t];
    const gmut<T> dst = to_global_mut(d.P) + (int64_t)r0 + 8 * w + g + (int64_t)(jb + 4 * c8) * ld;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int r = 8 * (q * NW + w) + g;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if ((int)(r < rows) & (int)(4 * c8 + t < ncb) & (int)(wg > 0 || r >= w32))
          dst[8 * q * NW + (int64_t)t * ld] = a[q][t] * vt[t];
    }
  }
  if (wg == 0 && w == NW - 1) t_factor(Gs, taus, to_global_mut(d.Tb) + (int64_t)jb * kNB);
}

// Block T factors for an existing reflector set (RRQR output): one workgroup
// per (descriptor, NB block).  G = V_b^T V_b on the matrix cores, the rows
// dealt to the waves 16 at a time (a lane reads four consecutive rows of two
// columns), summed in LDS; then one wave forms T from it.  Bound by latency:
// one pass over V_b and the T recurrence; a reduction per column of T took
// 160 us a launch at 64^3, 33^3 and 2-D alike.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_larft(const LarftDesc<T>* __restrict__ descs, const int* __restrict__ tstart,
                                                    int nd) {
  using V4 = typename Mfma<T>::v4;
  constexpr int NW = kThreads / kWave;
  __shared__ __align__(16) T Gs[kNB][kNB];
  __shared__ T part[NW][3][16][17];
  __shared__ T taus[kNB];
  const int t = blockIdx.x;
  const int p = find_owner(tstart, nd, t);
  const LarftDesc<T> d = descs[p];
  const int jb = (t - tstart[p]) * kNB;
  const int cols = min(kNB, d.r - jb), rows = d.m - jb;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave, c16 = lane & 15, k4 = lane >> 4;
  const int64_t ld = d.ldv;
  const gptr<T> V = to_global(d.V) + jb + (int64_t)jb * ld;
  if (tid < kNB) taus[tid] = tid < cols ? d.tau[jb + tid] : T(0);
  V4 g[3];  // tiles (0, 0), (0, 1), (1, 1) of G
#pragma unroll
  for (int q = 0; q < 3; ++q) g[q] = V4{T(0), T(0), T(0), T(0)};
  for (int rb = 16 * w; rb < rows; rb += 16 * NW) {
    T v[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = 16 * h + c16;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int r = rb + 4 * k4 + u;
        const bool in = (int)(r < rows) & (int)(c < cols);
        const T x = in ? V[r + (int64_t)c * ld] : T(0);
        v[h][u] = !in ? T(0) : (r > c ? x : (r == c ? T(1) : T(0)));
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      g[0] = Mfma<T>::mac(v[0][u], v[0][u], g[0]);
      g[1] = Mfma<T>::mac(v[0][u], v[1][u], g[1]);
      g[2] = Mfma<T>::mac(v[1][u], v[1][u], g[2]);
    }
  }
#pragma unroll
  for (int q = 0; q < 3; ++q)
#pragma unroll
    for (int u = 0; u < 4; ++u) part[w][q][Mfma<T>::row(k4, u)][c16] = g[q][u];
  __syncthreads();
  for (int e = tid; e < 3 * 256; e += kThreads) {
    const int q = e / 256, r = e / 16 % 16, c = e % 16;
    T s = part[0][q][r][c];
#pragma unroll
    for (int u = 1; u < NW; ++u) s += part[u][q][r][c];
    Gs[r + (q == 2 ? 16 : 0)][c + (q > 0 ? 16 : 0)] = s;
  }
  __syncthreads();
  if (w == 0) t_factor(Gs, taus, to_global_mut(d.Tb) + (int64_t)jb * kNB);
}

// B[:, jb:jb+w) <- B[:, jb:jb+w) * inv(R[jb:jb+w, jb:jb+w]) ; one row per thread.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_trsm_block(const TrsmDesc<T>* __restrict__ descs,
                                                         const int* __restrict__ tstart, int nd, int jb) {
  const int t = blockIdx.x;
  const int p = find_owner(tstart, nd, t);
  const TrsmDesc<T> d = descs[p];
  if (jb >= d.k) return;
  const int w = min(kNB, d.k - jb);
  __shared__ T Rs[kNB * kNB];
  for (int i = threadIdx.x; i < kNB * kNB; i += kThreads) {
    const int r = i % kNB, c = i / kNB;
    Rs[i] = (r < w && c < w) ? d.R[(jb + r) + (int64_t)(jb + c) * d.ldr] : T(0);
  }
  __syncthreads();
  const int row = (t - tstart[p]) * kThreads + threadIdx.x;
  if (row >= d.rows) return;
  T x[kNB];
#pragma unroll
  for (int c = 0; c < kNB; ++c) x[c] = (c < w) ? d.B[row + (int64_t)(jb + c) * d.ldb] : T(0);
#pragma unroll
  for (int c = 0; c < kNB; ++c) {
    if (c < w) {
      T s = x[c];
#pragma unroll
      for (int l = 0; l < kNB; ++l)
        if (l < c) s -= x[l] * Rs[l + c * kNB];
      x[c] = s / Rs[c + c * kNB];
    }
  }
#pragma unroll
  for (int c = 0; c < kNB; ++c)
    if (c < w) d.B[row + (int64_t)(jb + c) * d.ldb] = x[c];
}

int panel_nb() { return kNB; }
namespace {
// (waves, 8-row groups per lane), each holding 8 nw q rows in one workgroup;
// the last ones FP32 only.  A launch takes the first that holds its rows:
// launches of many small panels (more than kPanelCrowd; the scale phase of the
// lower levels has 670-6222) the fewest waves, whose redundant scalar work
// and barriers would fill the SIMDs, the others the most.  Panels of several
// workgroups take kPanelMulti: 512 rows a workgroup, as the exchange costs
// the same for 2 and 4 of them and a step is shorter than with 1280.
struct PanelForm { int nw, q, crowd; };
constexpr PanelForm kPanelForms[] = {{1, 4, 1},  {1, 8, 1},  {1, 16, 1}, {2, 16, 1}, {4, 4, 0},
                                     {4, 8, 0}, {8, 8, 0},  {8, 16, 0}, {8, 20, 0}, {8, 32, 0}};
constexpr int kNumPanelForms = sizeof(kPanelForms) / sizeof(kPanelForms[0]), kPanelCrowd = 512, kPanelMulti = 6;
template <typename T>
constexpr int panel_forms() { return sizeof(T) == 8 ? kNumPanelForms - 1 : kNumPanelForms; }

template <typename T>
int panel_form(int rows, int nd) {
  for (int f = 0; f < panel_forms<T>(); ++f)
    if (rows <= 8 * kPanelForms[f].nw * kPanelForms[f].q && (nd > kPanelCrowd || !kPanelForms[f].crowd)) return f;
  return panel_forms<T>() - 1;
}
template <typename T, int F>
const void* panel_fn(int f) {
  if constexpr (F < panel_forms<T>()) {
    if (f == F) return (const void*)k_panel_r<T, kPanelForms[F].nw, kPanelForms[F].q>;
    return panel_fn<T, F + 1>(f);
  } else {
    return nullptr;
  }
}
}  // namespace

template <typename T>
int panel_wgs(int rows) {
  constexpr PanelForm last = kPanelForms[panel_forms<T>() - 1], multi = kPanelForms[kPanelMulti];
  return rows <= 8 * last.nw * last.q ? 1 : (rows + 8 * multi.nw * multi.q - 1) / (8 * multi.nw * multi.q);
}
size_t panel_slots(int nwg) { return nwg > 1 ? (size_t)kNB * nwg * 2 * kNB : 0; }
template <typename T>
int panel_r_capacity() {
  const int f = kPanelMulti;
  int per_cu = 0, dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, panel_fn<T, 0>(f), kPanelForms[f].nw * kWave, 0) !=
      hipSuccess)
    return 0;
  return per_cu * cus;
}
// rows: the most rows [jb, m) of a panel of the launch; coop != 0 when a panel
// has several workgroups
template <typename T>
int launch_panel_r(hipStream_t s, const PanelDesc<T>* d, const int* wstart, int nd, int nwg_total, int jb, int rows,
                   int coop) {
  if (nd <= 0) return 0;
  const int f = coop ? kPanelMulti : panel_form<T>(rows, nd);
  const void* fn = panel_fn<T, 0>(f);
  void* args[] = {(void*)&d, (void*)&wstart, (void*)&nd, (void*)&jb};
  const dim3 block(kPanelForms[f].nw * kWave);
  if (!coop) return (int)hipLaunchKernel(fn, dim3(nwg_total), block, args, 0, s);
  return (int)launch_coresident(fn, dim3(nwg_total), block, args, 0, s);
}
template int panel_wgs<double>(int);
template int panel_wgs<float>(int);
template int panel_r_capacity<double>();
template int panel_r_capacity<float>();
template int launch_panel_r<double>(hipStream_t, const PanelDesc<double>*, const int*, int, int, int, int, int);
template int launch_panel_r<float>(hipStream_t, const PanelDesc<float>*, const int*, int, int, int, int, int);

template <typename T>
void launch_larft(hipStream_t s, const LarftDesc<T>* d, const int* tstart, int nd, int ntiles) {
  if (nd <= 0 || ntiles <= 0) return;
  hipLaunchKernelGGL((k_larft<T>), dim3(ntiles), dim3(kThreads), 0, s, d, tstart, nd);
}
template <typename T>
void launch_trsm_block(hipStream_t s, const TrsmDesc<T>* d, const int* tstart, int nd, int ntiles, int jb) {
  if (nd <= 0 || ntiles <= 0) return;
  hipLaunchKernelGGL((k_trsm_block<T>), dim3(ntiles), dim3(kThreads), 0, s, d, tstart, nd, jb);
}
int trsm_rows_per_tile() { return kThreads; }

template void launch_larft<double>(hipStream_t, const LarftDesc<double>*, const int*, int, int);
template void launch_larft<float>(hipStream_t, const LarftDesc<float>*, const int*, int, int);
template void launch_trsm_block<double>(hipStream_t, const TrsmDesc<double>*, const int*, int, int, int);
template void launch_trsm_block<float>(hipStream_t, const TrsmDesc<float>*, const int*, int, int, int);

}  // namespace spq
