// Kernel-level test entry points (libspaqr_ktest.so, loaded only by tests/).
// Each function uploads host arrays, runs one batched kernel family on the
// device and downloads the result, so single kernels can be checked against
// the oracle's LAPACK restatement.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "../kernels/descs.hpp"
#include "../kernels/launch.hpp"

using namespace spq;

namespace {
thread_local std::string g_err;
#define KT(call)                                                     \
  do {                                                               \
    hipError_t e_ = (call);                                          \
    if (e_ != hipSuccess) { g_err = hipGetErrorString(e_); return -1; } \
  } while (0)

// n elements on the device: the `given` of them that the caller's array has, then
// zeros
template <typename X>
X* dup(const X* h, size_t n, size_t given) {
  X* d = nullptr;
  if (hipMalloc((void**)&d, sizeof(X) * (n ? n : 1)) != hipSuccess) return nullptr;
  if (!h || given < std::max(n, size_t(1))) (void)hipMemset(d, 0, sizeof(X) * (n ? n : 1));
  if (h && given) (void)hipMemcpy(d, h, sizeof(X) * given, hipMemcpyHostToDevice);
  return d;
}
template <typename X>
X* dup(const X* h, size_t n) {
  return dup(h, n, n);
}
template <typename X>
void back(X* h, const X* d, size_t n) {
  if (n) (void)hipMemcpy(h, d, sizeof(X) * n, hipMemcpyDeviceToHost);
}
}  // namespace

extern "C" {

const char* ktest_last_error() { return g_err.c_str(); }

}  // extern "C"

namespace {
// C = alpha op(A) op(B) + beta C (single problem)
template <typename X>
int gemm_one(int m, int n, int k, const X* A, int lda, int acols, const X* B, int ldb, int bcols, X* Cm, int ldc,
             int flags, X alpha, X beta) {
  X *dA = dup(A, (size_t)lda * acols), *dB = dup(B, (size_t)ldb * bcols), *dC = dup(Cm, (size_t)ldc * n);
  GemmDesc<X> g{dA, dB, dC, lda, ldb, ldc, m, n, k, flags, alpha, beta};
  GemmDesc<X>* dg = dup(&g, 1);
  int tiles = gemm_tiles(m, n), zero = 0;
  int* ds = dup(&zero, 1);
  launch_gemm<X>(0, dg, ds, 1, tiles);
  KT(hipDeviceSynchronize());
  back(Cm, dC, (size_t)ldc * n);
  (void)hipFree(dA); (void)hipFree(dB); (void)hipFree(dC); (void)hipFree(dg); (void)hipFree(ds);
  return 0;
}
}  // namespace

extern "C" {

int ktest_gemm(int m, int n, int k, const double* A, int lda, int acols, const double* B, int ldb, int bcols,
               double* Cm, int ldc, int flags, double alpha, double beta) {
  return gemm_one<double>(m, n, k, A, lda, acols, B, ldb, bcols, Cm, ldc, flags, alpha, beta);
}
int ktest_gemm_f32(int m, int n, int k, const float* A, int lda, int acols, const float* B, int ldb, int bcols,
                   float* Cm, int ldc, int flags, float alpha, float beta) {
  return gemm_one<float>(m, n, k, A, lda, acols, B, ldb, bcols, Cm, ldc, flags, alpha, beta);
}

// Same product split along K into ksplit chunks (partials + ordered reduce).
int ktest_gemm_split(int m, int n, int k, const double* A, int lda, int acols, const double* B, int ldb, int bcols,
                     double* Cm, int ldc, int flags, double alpha, double beta, int ksplit) {
  if (ksplit < 1 || m < 1 || n < 1) { g_err = "bad split"; return -1; }
  double *dA = dup(A, (size_t)lda * acols), *dB = dup(B, (size_t)ldb * bcols), *dC = dup(Cm, (size_t)ldc * n);
  double* dW = dup<double>(nullptr, (size_t)ksplit * m * n);
  GemmDesc<double> g{dA, dB, dC, lda, ldb, ldc, m, n, k, flags, alpha, beta, ksplit, dW};
  GemmDesc<double>* dg = dup(&g, 1);
  int zero = 0;
  int* ds = dup(&zero, 1);
  launch_gemm<double>(0, dg, ds, 1, gemm_tiles(m, n) * ksplit);
  if (ksplit > 1) launch_gemm_reduce<double>(0, dg, ds, 1, (m * n + 255) / 256);
  KT(hipDeviceSynchronize());
  back(Cm, dC, (size_t)ldc * n);
  (void)hipFree(dA); (void)hipFree(dB); (void)hipFree(dC); (void)hipFree(dW); (void)hipFree(dg); (void)hipFree(ds);
  return 0;
}

// sigma_min of upper-triangular R (k x k, ld) by the Lanczos kernel.
int ktest_smin(int k, const double* R, int ld, double* out) {
  if (k < 1 || k > smin_max_k() || ld < k) { g_err = "bad smin shape"; return -1; }
  double* dR = dup(R, (size_t)ld * k);
  double* dW = dup<double>(nullptr, smin_work_elems(k));
  double* dO = dup<double>(nullptr, 1);
  SminDesc<double> sd{dR, ld, k, dW, dO};
  SminDesc<double>* dd = dup(&sd, 1);
  launch_smin<double>(0, dd, 1, k);
  KT(hipDeviceSynchronize());
  back(out, dO, 1);
  (void)hipFree(dR); (void)hipFree(dW); (void)hipFree(dO); (void)hipFree(dd);
  return 0;
}

}  // extern "C"
namespace {
// Blocked Householder QR of one m x k panel (col-major, ld m): A <- V\R,
// tau (min(m,k)), Tb (nb x roundup(k,nb)), and C (m x nc) <- Q^T C.
template <typename X>
int qr_one(int m, int k, X* A, X* tau, X* Tb, int nc, X* Cm) {
  const int nb = panel_nb(), kk = m < k ? m : k, nblk = (k + nb - 1) / nb;
  X *dA = dup(A, (size_t)m * k), *dt = dup<X>(nullptr, k), *dT = dup<X>(nullptr, (size_t)nb * nb * nblk);
  X* dC = dup(Cm, (size_t)m * (nc > 0 ? nc : 1), (size_t)m * nc);
  int zero = 0;
  int* ds = dup(&zero, 1);
  int* err = dup<int>(nullptr, 1);
  for (int jb = 0; jb < kk; jb += nb) {
    const int nwg = panel_wgs<X>(m - jb);
    if (nwg > panel_r_capacity<X>()) { g_err = "nwg exceeds resident capacity"; return -1; }
    X* part = dup<X>(nullptr, panel_slots(nwg));
    PanelDesc<X> pd{dA, dt, dT, m, m, k, nwg, part, err};
    PanelDesc<X>* dpd = dup(&pd, 1);
    const int rc = launch_panel_r<X>(0, dpd, ds, 1, nwg, jb, m - jb, nwg > 1 ? 1 : 0);
    if (rc != 0) { g_err = hipGetErrorString((hipError_t)rc); return -1; }
    KT(hipDeviceSynchronize());
    for (void* q : {(void*)part, (void*)dpd}) (void)hipFree(q);
    const int w = (nb < kk - jb) ? nb : kk - jb, rows = m - jb;
    const X* Vb = dA + jb + (size_t)jb * m;
    const X* Tbb = dT + (size_t)jb * nb;
    // the engine's descriptors for this step (W = V_b T_b^T, Y = V_b^T C,
    // C -= W Y), each list run as one batched launch as the engine does
    std::vector<LarfbTarget<X>> tg;
    const int c0 = jb + ((nb < k - jb) ? nb : k - jb);
    if (k > c0) tg.push_back({dA + jb + (size_t)c0 * m, m, k - c0});
    if (nc > 0) tg.push_back({dC + jb, m, nc});
    std::vector<void*> scratch;
    auto alloc = [&](int64_t elems) {
      X* p = dup<X>(nullptr, (size_t)(elems > 0 ? elems : 1));
      scratch.push_back(p);
      return p;
    };
    std::vector<GemmDesc<X>> g1, g3;
    larfb_step_descs<X>(Vb, m, Tbb, nb, rows, w, tg.data(), (int)tg.size(), alloc, g1, g3);
    for (auto* gl : {&g1, &g3}) {
      if (gl->empty()) continue;
      std::vector<int> st(gl->size());
      int nt = 0;
      for (size_t i = 0; i < gl->size(); ++i) { st[i] = nt; nt += gemm_tiles((*gl)[i].m, (*gl)[i].n); }
      GemmDesc<X>* dg = dup(gl->data(), gl->size());
      int* dst = dup(st.data(), st.size());
      launch_gemm<X>(0, dg, dst, (int)gl->size(), nt);
      KT(hipDeviceSynchronize());
      (void)hipFree(dg);
      (void)hipFree(dst);
    }
    for (void* p : scratch) (void)hipFree(p);
  }
  KT(hipDeviceSynchronize());
  back(A, dA, (size_t)m * k);
  back(tau, dt, kk);
  back(Tb, dT, (size_t)nb * nb * nblk);
  if (nc > 0) back(Cm, dC, (size_t)m * nc);
  int e = 0;
  back(&e, err, 1);
  for (void* p : {(void*)dA, (void*)dt, (void*)dT, (void*)dC, (void*)ds, (void*)err}) (void)hipFree(p);
  if (e) { g_err = "barrier wait timed out"; return -1; }
  return 0;
}

// Block T factors of V (m x r) and tau.
template <typename X>
int larft_one(int m, int r, const X* V, const X* tau, X* Tb) {
  const int nb = panel_nb(), nblk = (r + nb - 1) / nb;
  X *dV = dup(V, (size_t)m * r), *dt = dup(tau, r), *dT = dup<X>(nullptr, (size_t)nb * nb * nblk);
  LarftDesc<X> d{dV, dt, dT, m, m, r, 0};
  LarftDesc<X>* dd = dup(&d, 1);
  int zero = 0;
  int* ds = dup(&zero, 1);
  launch_larft<X>(0, dd, ds, 1, nblk);
  KT(hipDeviceSynchronize());
  back(Tb, dT, (size_t)nb * nb * nblk);
  for (void* p : {(void*)dV, (void*)dt, (void*)dT, (void*)dd, (void*)ds}) (void)hipFree(p);
  return 0;
}
}  // namespace
extern "C" {
int ktest_qr(int m, int k, double* A, double* tau, double* Tb, int nc, double* Cm) {
  return qr_one<double>(m, k, A, tau, Tb, nc, Cm);
}
int ktest_qr_f32(int m, int k, float* A, float* tau, float* Tb, int nc, float* Cm) {
  return qr_one<float>(m, k, A, tau, Tb, nc, Cm);
}
int ktest_larft(int m, int r, const double* V, const double* tau, double* Tb) {
  return larft_one<double>(m, r, V, tau, Tb);
}
int ktest_larft_f32(int m, int r, const float* V, const float* tau, float* Tb) {
  return larft_one<float>(m, r, V, tau, Tb);
}

// Truncated QP3 of C (k x N): Ct is N x k (ld N) in/out; V k x k, tau k.
// form 0: streaming kernel split over nwg workgroups; form 1 / 2: register
// kernel with 256 / 1024-thread workgroups and 32 rows per lane; form
// 10 * rc + 1 / 2: the same with rc rows per lane (group size and workgroup
// count follow from k and N).  Multi-
// workgroup problems are launched cooperatively.  Returns the rank, or -1 on
// a launch/run error.
int ktest_qp3(int k, int N, double* Ct, double* V, double* tau, double tol, int nwg, int form) {
  int G = 0, nt = 256;
  const int rcv = form >= 10 ? form / 10 : 32;  // register form rows per lane
  if (form >= 1) {
    G = qp3r_lanes(k, rcv);
    if (G == 0) { g_err = "k too large for the register form"; return -1; }
    nt = (form % 10) == 2 ? 1024 : 256;
    nwg = (N + nt / G - 1) / (nt / G);
    if (nwg > qp3r_capacity<double>(G, nt, rcv)) { g_err = "nwg exceeds resident capacity"; return -1; }
  } else if (nwg > qp3_capacity<double>(k)) {
    g_err = "nwg exceeds resident capacity";
    return -1;
  }
  double *dC = dup(Ct, (size_t)N * k), *dV = dup<double>(nullptr, (size_t)k * k), *dt = dup<double>(nullptr, k);
  double* vn = dup<double>(nullptr, 2 * (size_t)N);
  int* pos = dup<int>(nullptr, 2 * (size_t)N * nwg);
  double* pv = dup<double>(nullptr, 4 * (size_t)nwg);
  int* pp = dup<int>(nullptr, 4 * (size_t)nwg);
  double* beta = dup<double>(nullptr, k);
  unsigned int* sync = dup<unsigned int>(nullptr, barrier_words(nwg));
  int* err = dup<int>(nullptr, 1);
  int* rk = dup<int>(nullptr, 1);
  double* pcol = dup<double>(nullptr, 2 * (size_t)nwg * std::max(k, G * rcv));
  Qp3Desc<double> d{dC, dV, dt, vn, pos, pv, pp, beta, sync, err, rk, pcol, N, k, N, k, tol, nwg, G, rcv};
  Qp3Desc<double>* dd = dup(&d, 1);
  int zero = 0;
  int* ws = dup(&zero, 1);
  int rc = form >= 1 ? launch_qp3r<double>(0, dd, ws, 1, nwg, G, N, nt, rcv, nwg > 1 ? 1 : 0)
                     : launch_qp3<double>(0, dd, ws, 1, nwg, k, nwg > 1 ? 1 : 0);
  if (rc != 0) { g_err = hipGetErrorString((hipError_t)rc); return -1; }
  KT(hipDeviceSynchronize());
  int rank = 0, e = 0;
  back(&rank, rk, 1);
  back(&e, err, 1);
  back(Ct, dC, (size_t)N * k);
  back(V, dV, (size_t)k * k);
  back(tau, dt, k);
  for (void* q : {(void*)dC, (void*)dV, (void*)dt, (void*)vn, (void*)pos, (void*)pv, (void*)pp, (void*)beta,
                  (void*)sync, (void*)err, (void*)rk, (void*)dd, (void*)ws, (void*)pcol})
    (void)hipFree(q);
  if (e) { g_err = "barrier wait timed out"; return -1; }
  return rank;
}

// The same by the blocked form (rounds of a panel and an update launch) in T
// storage.  Returns the rank (rounds in *rounds), or -1.
}  // extern "C"
namespace {
template <typename X>
int rrqr_one(int k, int N, X* Ct, X* V, X* tau, double tol, int nd, int* perm, int* rounds) {
  const int form = rrqr_form(k, nd);  // the form a launch of nd problems takes
  if (!form || k < 1 || N < 0) { g_err = "k beyond the blocked form"; return -1; }
  const size_t n1 = std::max(N, 1);
  const int ldv = k + kRrqrPivots - 1, kr = k + 15;  // V by rows, padded
  X *dC = dup(Ct, n1 * k, (size_t)N * k), *dV = dup<X>(nullptr, (size_t)kr * ldv), *dt = dup<X>(nullptr, k);
  double* tm = dup<double>(nullptr, kRrqrPivots * kRrqrPivots);
  double* vn = dup<double>(nullptr, n1);
  int *ip = dup<int>(nullptr, n1), *pm = dup<int>(nullptr, n1);
  RrqrState* st = dup<RrqrState>(nullptr, 1);
  RrqrDesc<X> d{dC, dV, dt, tm, vn, ip, pm, st, (int)n1, k, N, ldv, tol};
  RrqrDesc<X>* dd = dup(&d, 1);
  int zero = 0;
  int* ws = dup(&zero, 1);
  launch_rrqr_init<X>(0, dd, ws, 1, rrqr_init_tiles(N));
  RrqrState h{};
  int r = 0;
  for (; r <= k; ++r) {
    launch_rrqr_panel<X>(0, dd, 1, form);
    launch_rrqr_update<X>(0, dd, ws, 1, ((int)n1 + rrqr_update_cols() - 1) / rrqr_update_cols(), k);
    KT(hipDeviceSynchronize());
    back(&h, st, 1);
    if (h.done) break;
  }
  std::vector<X> hv((size_t)kr * ldv);
  back(Ct, dC, (size_t)N * k);
  back(hv.data(), dV, hv.size());
  for (int c = 0; c < k; ++c)
    for (int i = 0; i < k; ++i) V[i + (size_t)c * k] = hv[(size_t)i * ldv + c];
  back(tau, dt, k);
  back(perm, pm, N);
  *rounds = r + 1;
  for (void* q : {(void*)dC, (void*)dV, (void*)dt, (void*)tm, (void*)vn, (void*)ip, (void*)pm, (void*)st,
                  (void*)dd, (void*)ws})
    (void)hipFree(q);
  if (!h.done) { g_err = "no progress"; return -1; }
  return h.next;
}
}  // namespace
namespace {
template <typename T>
int larfb_one(int form, int rows, int cols, int nt, int w, const T* V, int ldv, const T* Tb, T* Cm, int ldc) {
  if (form < 0 || form >= larfb_forms() || rows > larfb_form_rows(form)) { g_err = "rows exceed the form"; return -1; }
  T *dV = dup(V, (size_t)ldv * w), *dT = dup(Tb, 32 * 32), *dC = dup(Cm, (size_t)ldc * cols * nt);
  std::vector<LarfbDesc<T>> ds;
  std::vector<int> st{0};
  for (int t = 0; t < nt; ++t) {
    ds.push_back(LarfbDesc<T>{dV, dT, dC + (size_t)ldc * cols * t, ldv, ldc, rows, cols, w, 0});
    st.push_back(st.back() + larfb_tiles(cols));
  }
  launch_larfb<T>(0, dup(ds.data(), ds.size()), dup(st.data(), st.size()), nt, st.back(), form);
  KT(hipDeviceSynchronize());
  back(Cm, dC, (size_t)ldc * cols * nt);
  return 0;
}
}  // namespace
namespace {
// One dataflow op (kernels/flow.hip) on x (m values) and, for the triangular
// and the pull form, xn (n values) with the block Bn: the inputs lie in two
// segments (or `pieces`) in reverse order, the blocks' tiles start with a short
// one.
//   WY: A, B m x k (lda, ldb), parts of rows_per rows; unit: A is V, B is W
//   Back: R = A (k x k, m = k), Bn k x n (ldb), nwg parts; SolveT: R alone
//   Pull: Bn = B n x m (ldb)
template <typename T>
int flow_one(int type, int m, int k, int par, int unit, const T* A, int lda, const T* B, int ldb, int n,
             const double* x, const double* xn, double* out, int pieces = 0) {
  const int total = 2 * m + n + 7;
  std::vector<int> cut{0};
  if (pieces)
    for (int p = 1; p <= pieces; ++p) cut.push_back((int)((int64_t)m * p / pieces));
  else
    for (int e : {m - m / 3, m}) cut.push_back(e);
  std::vector<FlowSeg> segs;
  std::vector<double> xin(m + n);
  for (size_t p = 0; p + 1 < cut.size(); ++p) {
    const int len = cut[p + 1] - cut[p], off = m - cut[p + 1];  // the last rows lie first
    if (len > 0) segs.push_back(FlowSeg{off, len});
    for (int i = 0; i < len; ++i) xin[off + i] = x[cut[p] + i];
  }
  if ((int)segs.size() > kFlowMaxSegs) { g_err = "too many segments"; return -1; }
  for (int i = 0; i < n; ++i) xin[m + i] = xn[i];
  const bool tri = type == kFlowBack || type == kFlowSolveT, wy = type == kFlowWY;
  T* dA = A ? dup(A, (size_t)lda * k) : nullptr;
  T* dB = B ? dup(B, (size_t)ldb * (wy ? k : (type == kFlowPull ? m : n))) : nullptr;
  std::vector<FlowBlk<T>> blks;
  if (type == kFlowBack)
    for (int j = 0; j < n;) {
      const int w = std::min(j == 0 ? 5 : 32, n - j);
      blks.push_back(FlowBlk<T>{dB + (size_t)j * ldb, ldb, w, m + j, 0});
      j += w;
    }
  if (type == kFlowPull)
    for (int r = 0; r < n;) {
      const int w = std::min(r == 0 ? 7 : 64, n - r);
      blks.push_back(FlowBlk<T>{dB + r, ldb, w, m + r, 0});
      r += w;
    }
  FlowOp<T> d{};
  d.type = type; d.m = m; d.k = wy || tri ? k : 32;
  d.A = dA; d.lda = lda; d.B = dB; d.ldb = ldb;
  d.unit_a = unit; d.unit_b = !unit;
  d.rows_per = par;
  d.nwg = wy ? (m + par - 1) / par : (tri ? par : 1);
  d.nseg = (int)segs.size(); d.nblk = (int)blks.size(); d.out = m + n + 7;
  const int nb = (k + 31) / 32, np = type == kFlowPull ? (m + 31) / 32 : d.nwg;
  d.slots = dup<T>(nullptr, (size_t)d.nwg * d.k);
  T* dx = dup<T>(nullptr, total);
  unsigned int* ctl = dup<unsigned int>(nullptr, 64);
  int* err = dup<int>(nullptr, 64);
  if (tri) {
    T* D = dup<T>(nullptr, flow_diag_elems(k));
    FlowDiag<T> fd{dA, D, lda, k, type == kFlowSolveT, 0};
    const int st[2] = {0, nb};
    launch_flow_diag<T>(0, dup(&fd, 1), dup(st, 2), 1, nb);
    d.B = D;
  }
  std::vector<FlowOp<T>> parts;
  for (int g = 0; g < np; ++g) { d.g = g; parts.push_back(d); }
  FlowArgs<T> a{};
  a.parts = dup(parts.data(), parts.size());
  a.segs = dup(segs.data(), segs.size());
  a.blks = blks.empty() ? nullptr : dup(blks.data(), blks.size());
  a.x = dx; a.ctl = ctl; a.err = err; a.nparts = np;
  launch_flow_begin<T>(0, nullptr, m + n, dup(xin.data(), xin.size()), dx, 0, FlowClear{});
  launch_flow<T>(0, a, std::min(np, flow_capacity<T>()));
  std::vector<int> loc(m);
  for (int i = 0; i < m; ++i) loc[i] = d.out + i;
  double* dy = dup<double>(nullptr, m);
  launch_flow_out<T>(0, dup(loc.data(), loc.size()), m, dx, nullptr, dy);
  KT(hipMemcpy(out, dy, sizeof(double) * m, hipMemcpyDeviceToHost));
  int e = 0;
  KT(hipMemcpy(&e, err, sizeof(int), hipMemcpyDeviceToHost));
  return e;
}
}  // namespace
extern "C" {
int ktest_flow(int type, int m, int k, int par, int unit, const double* A, int lda, const double* B, int ldb, int n,
               const double* x, const double* xn, double* out) {
  return flow_one<double>(type, m, k, par, unit, A, lda, B, ldb, n, x, xn, out);
}
int ktest_flow_pieces(int pieces, int type, int m, int k, int par, int unit, const double* A, int lda, const double* B,
                      int ldb, int n, const double* x, const double* xn, double* out) {
  return flow_one<double>(type, m, k, par, unit, A, lda, B, ldb, n, x, xn, out, pieces);
}
// One k_larfb step of `form` on nt targets of cols columns each (C: ldc x nt
// cols, target t at its column t cols)
int ktest_larfb(int form, int rows, int cols, int nt, int w, const double* V, int ldv, const double* Tb, double* Cm,
                int ldc) {
  return larfb_one<double>(form, rows, cols, nt, w, V, ldv, Tb, Cm, ldc);
}
int ktest_larfb_f32(int form, int rows, int cols, int nt, int w, const float* V, int ldv, const float* Tb, float* Cm,
                    int ldc) {
  return larfb_one<float>(form, rows, cols, nt, w, V, ldv, Tb, Cm, ldc);
}
int ktest_larfb_rows(int form) { return form < larfb_forms() ? larfb_form_rows(form) : 0; }
int ktest_flow_f32(int type, int m, int k, int par, int unit, const float* A, int lda, const float* B, int ldb, int n,
                   const double* x, const double* xn, double* out) {
  return flow_one<float>(type, m, k, par, unit, A, lda, B, ldb, n, x, xn, out);
}
int ktest_rrqr(int k, int N, double* Ct, double* V, double* tau, double tol, int nd, int* perm, int* rounds) {
  return rrqr_one<double>(k, N, Ct, V, tau, tol, nd, perm, rounds);
}
int ktest_rrqr_f32(int k, int N, float* Ct, float* V, float* tau, double tol, int nd, int* perm, int* rounds) {
  return rrqr_one<float>(k, N, Ct, V, tau, tol, nd, perm, rounds);
}

// Timing of one truncated QP3 problem (either form): `reps` launches on a
// fresh copy of C each, the average kernel time in *ms.  Returns the rank.
int ktest_qp3_bench(int k, int N, const double* Ct, double tol, int form, int nwg, int reps, double* ms) {
  int G = 0, nt = 256;
  const int rcv = form >= 10 ? form / 10 : 32;  // register form rows per lane
  if (form >= 1) {
    G = qp3r_lanes(k, rcv);
    if (G == 0) { g_err = "k too large for the register form"; return -1; }
    nt = (form % 10) == 2 ? 1024 : 256;
    nwg = (N + nt / G - 1) / (nt / G);
    if (nwg > qp3r_capacity<double>(G, nt, rcv)) { g_err = "nwg exceeds resident capacity"; return -1; }
  } else if (nwg > qp3_capacity<double>(k)) {
    g_err = "nwg exceeds resident capacity";
    return -1;
  }
  double *d0 = dup(Ct, (size_t)N * k), *dC = dup<double>(nullptr, (size_t)N * k);
  double *dV = dup<double>(nullptr, (size_t)k * k), *dt = dup<double>(nullptr, k);
  double* vn = dup<double>(nullptr, 2 * (size_t)N);
  int* pos = dup<int>(nullptr, 2 * (size_t)N * nwg);
  double* pv = dup<double>(nullptr, 4 * (size_t)nwg);
  int* pp = dup<int>(nullptr, 4 * (size_t)nwg);
  double* beta = dup<double>(nullptr, k);
  unsigned int* sync = dup<unsigned int>(nullptr, barrier_words(nwg));
  int* err = dup<int>(nullptr, 1);
  int* rk = dup<int>(nullptr, 1);
  double* pcol = dup<double>(nullptr, 2 * (size_t)nwg * std::max(k, G * rcv));
  Qp3Desc<double> d{dC, dV, dt, vn, pos, pv, pp, beta, sync, err, rk, pcol, N, k, N, k, tol, nwg, G, rcv};
  Qp3Desc<double>* dd = dup(&d, 1);
  int zero = 0;
  int* ws = dup(&zero, 1);
  hipEvent_t a, b;
  KT(hipEventCreate(&a));
  KT(hipEventCreate(&b));
  double tot = 0;
  int rc = 0;
  for (int r = 0; r < reps && rc == 0; ++r) {
    KT(hipMemcpy(dC, d0, sizeof(double) * (size_t)N * k, hipMemcpyDeviceToDevice));
    KT(hipMemset(sync, 0, sizeof(unsigned int) * barrier_words(nwg)));
    KT(hipEventRecord(a, 0));
    rc = form >= 1 ? launch_qp3r<double>(0, dd, ws, 1, nwg, G, N, nt, rcv, nwg > 1 ? 1 : 0)
                   : launch_qp3<double>(0, dd, ws, 1, nwg, k, nwg > 1 ? 1 : 0);
    KT(hipEventRecord(b, 0));
    KT(hipEventSynchronize(b));
    float t = 0;
    KT(hipEventElapsedTime(&t, a, b));
    tot += t;
  }
  if (rc != 0) { g_err = hipGetErrorString((hipError_t)rc); return -1; }
  *ms = tot / reps;
  int rank = 0, e = 0;
  back(&rank, rk, 1);
  back(&e, err, 1);
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  for (void* q : {(void*)d0, (void*)dC, (void*)dV, (void*)dt, (void*)vn, (void*)pos, (void*)pv, (void*)pp,
                  (void*)beta, (void*)sync, (void*)err, (void*)rk, (void*)dd, (void*)ws, (void*)pcol})
    (void)hipFree(q);
  if (e) { g_err = "barrier wait timed out"; return -1; }
  return rank;
}

// x <- H^T x (trans=1) or H x for blocked reflectors (V m x k, Tb), with x
// split into `nseg` equal-length segments stored at stride `gap` in a buffer.
// form 0: LDS form (4 row-slice workgroups for m >= 2048); form 1: register
// form, 7 row waves (ceil(m / 448) workgroups); form 2: register form with
// the row waves reflr_row_waves(m) gives (1 or 2 for m <= 128, else 7)
int ktest_refl(int m, int k, const double* V, const double* Tb, double* x, int trans, int nseg, int gap, int form) {
  const int nb = panel_nb(), nblk = (k + nb - 1) / nb;
  const int seglen = m / nseg;
  const size_t xlen = (size_t)nseg * (seglen + gap);
  double *dV = dup(V, (size_t)m * k), *dT = dup(Tb, (size_t)nb * nb * nblk);
  std::vector<double> xb(xlen, -7.0);
  std::vector<Seg> segs;
  for (int s = 0; s < nseg; ++s) {
    segs.push_back(Seg{(int64_t)s * (seglen + gap), seglen, 0});
    std::memcpy(&xb[(size_t)s * (seglen + gap)], x + (size_t)s * seglen, sizeof(double) * seglen);
  }
  double* dx = dup(xb.data(), xlen);
  Seg* dsg = dup(segs.data(), segs.size());
  const int nrw = form == 2 ? reflr_row_waves(m) : 7;
  const int nwg = form ? (m + 64 * nrw - 1) / (64 * nrw) : (m >= 2048 ? 4 : 1);
  double* wk = dup<double>(nullptr, m);
  double* part = dup<double>(nullptr, 2 * 32 * (size_t)nwg);
  unsigned int* sync = dup<unsigned int>(nullptr, 1);
  int* err = dup<int>(nullptr, 1);
  ReflDesc<double> d{dV, dT, m, m, k, nb, 0, nseg, trans, nwg, wk, part, sync, err};
  ReflDesc<double>* dd = dup(&d, 1);
  double* work = dup<double>(nullptr, m);
  int zero = 0;
  int* ws = dup(&zero, 1);
  if (form) launch_reflr<double>(0, dd, ws, 1, nwg, dsg, dx, nseg, nrw);
  else launch_refl<double>(0, dd, ws, 1, nwg, dsg, dx, work, nwg > 1 ? 0 : m);
  KT(hipDeviceSynchronize());
  back(xb.data(), dx, xlen);
  for (int s = 0; s < nseg; ++s)
    std::memcpy(x + (size_t)s * seglen, &xb[(size_t)s * (seglen + gap)], sizeof(double) * seglen);
  int e = 0;
  back(&e, err, 1);
  for (void* p : {(void*)dV, (void*)dT, (void*)dx, (void*)dsg, (void*)dd, (void*)work, (void*)wk, (void*)part,
                  (void*)sync, (void*)err, (void*)ws})
    (void)hipFree(p);
  if (e) { g_err = "barrier wait timed out"; return -1; }
  return 0;
}

// xs <- R^{-1}(xs - A1 x1) (trans=0) ; or xs <- R^{-T} xs, x1 -= A1^T xs (trans=1)
// form 1: the latency form (one workgroup, no R12 products: s must be 0)
int ktest_bwd(int k, const double* R, int s, const double* A1, double* xs, double* x1, int trans, int form) {
  double *dR = dup(R, (size_t)k * k), *dA = dup(A1, (size_t)k * (s > 0 ? s : 1), (size_t)k * s);
  std::vector<double> xb((size_t)k + s);
  std::memcpy(xb.data(), xs, sizeof(double) * k);
  if (s > 0) std::memcpy(xb.data() + k, x1, sizeof(double) * s);
  double* dx = dup(xb.data(), xb.size());
  R12Desc<double> q{dA, k, s, (int64_t)k};
  R12Desc<double>* dq = dup(&q, 1);
  const int nwg = k >= 512 ? 4 : 1;
  unsigned int* sync = dup<unsigned int>(nullptr, 1);
  int* err = dup<int>(nullptr, 1);
  BwdDesc<double> d{dR, k, k, 0, 0, s > 0 ? 1 : 0, trans, nwg, sync, err};
  BwdDesc<double>* dd = dup(&d, 1);
  int zero = 0;
  int* ws = dup(&zero, 1);
  if (form) {
    BwdDesc<double> d1 = d;
    d1.nwg = 1;
    KT(hipMemcpy(dd, &d1, sizeof(d1), hipMemcpyHostToDevice));
    launch_bwdr<double>(0, dd, 1, k, dx);
  } else {
    launch_bwd<double>(0, dd, ws, 1, nwg, dq, dx);
  }
  KT(hipDeviceSynchronize());
  back(xb.data(), dx, xb.size());
  std::memcpy(xs, xb.data(), sizeof(double) * k);
  if (s > 0) std::memcpy(x1, xb.data() + k, sizeof(double) * s);
  int e = 0;
  back(&e, err, 1);
  for (void* p : {(void*)dR, (void*)dA, (void*)dx, (void*)dq, (void*)dd, (void*)sync, (void*)err, (void*)ws})
    (void)hipFree(p);
  if (e) { g_err = "barrier wait timed out"; return -1; }
  return 0;
}

// B (rows x k) <- B R^{-1} with the blocked GEMM + row-block solve.
int ktest_trsm(int rows, int k, const double* R, double* B) {
  const int nb = panel_nb();
  double *dR = dup(R, (size_t)k * k), *dB = dup(B, (size_t)rows * k);
  int zero = 0;
  int* ds = dup(&zero, 1);
  for (int jb = 0; jb < k; jb += nb) {
    const int w = (nb < k - jb) ? nb : k - jb;
    if (jb > 0) {
      GemmDesc<double> g{dB, dR + (size_t)jb * k, dB + (size_t)jb * rows, rows, k, rows, rows, w, jb,
                         gemm_flags(false, false), -1.0, 1.0};
      GemmDesc<double>* dg = dup(&g, 1);
      launch_gemm<double>(0, dg, ds, 1, gemm_tiles(rows, w));
      KT(hipDeviceSynchronize());
      (void)hipFree(dg);
    }
    TrsmDesc<double> t{dB, dR, rows, k, rows, k};
    TrsmDesc<double>* dt = dup(&t, 1);
    launch_trsm_block<double>(0, dt, ds, 1, (rows + trsm_rows_per_tile() - 1) / trsm_rows_per_tile(), jb);
    KT(hipDeviceSynchronize());
    (void)hipFree(dt);
  }
  back(B, dB, (size_t)rows * k);
  for (void* p : {(void*)dR, (void*)dB, (void*)ds}) (void)hipFree(p);
  return 0;
}

// Batched copy round trip: dst = src (trans 0/1) for one block.
int ktest_copy(int rows, int cols, const double* src, int lds, double* dst, int ldd, int trans) {
  const int drows = trans ? cols : rows, dcols = trans ? rows : cols;
  double *ds_ = dup(src, (size_t)lds * cols), *dd = dup(dst, (size_t)ldd * dcols);
  CopyDesc c{ds_, dd, lds, ldd, rows, cols, trans, 0};
  CopyDesc* dc = dup(&c, 1);
  int zero = 0;
  int* st = dup(&zero, 1);
  launch_copy(0, 8, 8, dc, st, 1, ((rows + 31) / 32) * ((cols + 31) / 32));
  KT(hipDeviceSynchronize());
  back(dst, dd, (size_t)ldd * dcols);
  (void)drows;
  for (void* p : {(void*)ds_, (void*)dd, (void*)dc, (void*)st}) (void)hipFree(p);
  return 0;
}

}  // extern "C"
