// Host code of the engine against the runtime of fake_hip.hpp, where what the
// device would read, and memory that has run out, can be looked at.  One case per
// argument; exit code 0 and "ok" when it holds.
#define private public
#include "engine.cpp"
#undef private
#include "fake_hip.hpp"

using namespace spq;

// ---- launchers the cases reach
namespace seen {
const void* flow_x = nullptr;  // of the last apply
int flow_begins = 0, flow_parts = 0, panel_calls = 0;
void (*on_panel)(const RrqrDesc<double>*, int) = nullptr;
}  // namespace seen
namespace spq {
void host_prof_start() {}
int panel_nb() { return 32; }
int refl_lds_cap(int) { return 1 << 20; }
int bwdr_max_k() { return 1 << 20; }
int reflr_rows() { return 448; }
int r12_chunk_cols() { return 64; }
int reflr_row_waves(int) { return 7; }
size_t reflr_lds(int) { return 0; }
size_t flow_diag_elems(int k) { return (size_t)((k + 31) / 32) * 32 * 33; }
template <> int flow_capacity<double>() { return 512; }
template <> int flow_capacity<float>() { return 512; }
void launch_zero(hipStream_t, int elem, void* p, int64_t n) { std::memset(p, 0, (size_t)elem * (size_t)n); }
template <> void launch_flow_diag<double>(hipStream_t, const FlowDiag<double>*, const int*, int, int) {}
template <> void launch_gemm<double>(hipStream_t, const GemmDesc<double>*, const int*, int, int) {}
template <> void launch_flow_begin<double>(hipStream_t, const int*, int, const double*, double* x, int, const FlowClear&) {
  CHECK(x);
  seen::flow_x = x;
  ++seen::flow_begins;
}
template <> void launch_flow<double>(hipStream_t, const FlowArgs<double>& a, int grid) {
  CHECK(a.x == seen::flow_x && a.nparts > 0 && a.parts && a.segs && a.ctl && a.err && grid > 0);
  seen::flow_parts = a.nparts;
}
template <> void launch_flow_out<double>(hipStream_t, const int* at, int n, const double* x, const int*, double*) {
  CHECK(at && x == seen::flow_x && n > 0);
}
int rrqr_form(int k, int) { return k <= 704 ? 1 : 0; }
int rrqr_form_waves(int f) { return f == 1 ? 1 : 0; }
int rrqr_form_rows(int f) { return f == 1 ? 16 : 0; }
int rrqr_init_tiles(int) { return 1; }
int rrqr_update_cols() { return 16; }
template <> void launch_rrqr_init<double>(hipStream_t, const RrqrDesc<double>* d, const int*, int nd, int) {
  for (int q = 0; q < nd; ++q) *d[q].st = RrqrState{};
}
template <> void launch_rrqr_panel<double>(hipStream_t, const RrqrDesc<double>* d, int nd, int) {
  ++seen::panel_calls;
  if (seen::on_panel) seen::on_panel(d, nd);
}
template <> void launch_rrqr_update<double>(hipStream_t, const RrqrDesc<double>*, const int*, int, int, int) {}
}  // namespace spq

namespace {
CscMat grid(int n) {  // 5-point pattern
  CscMat A;
  A.m = A.n = n * n;
  A.p.push_back(0);
  for (int j = 0; j < n * n; ++j) {
    const int x = j % n, y = j / n;
    for (int d : {-n, -1, 0, 1, n}) {
      if ((d == -n && y == 0) || (d == n && y == n - 1) || (d == -1 && x == 0) || (d == 1 && x == n - 1)) continue;
      A.i.push_back(j + d);
      A.x.push_back(d == 0 ? 4.0 : -1.0);
    }
    A.p.push_back((int)A.i.size());
  }
  return A;
}

// a partitioned tree with the ops of an elimination of its leaves
struct Made {
  Engine<double> e;
  std::vector<double> factors;
  explicit Made(int n = 16, int nlevels = 3) : e(nlevels, 0, 0), factors(1 << 16) {
    e.set_square(1);
    e.set_coords(tensor_coordinates(n, 2), 2);
    e.partition(grid(n));
    for (int c : e.bottoms_[0]) {
      const int k = e.cl_[c].rsize;
      if (k <= 0) continue;
      Engine<double>::Op o{};
      o.kind = Engine<double>::OpQR;
      o.level = 0;
      o.c = c;
      o.V = o.Tb = o.R = factors.data();
      o.ldv = o.m = o.k = o.ldr = o.kr = k;
      o.segs.push_back({c, k});
      e.ops_.push_back(o);
      e.alloc_x(c, k);
    }
    CHECK(!e.ops_.empty());
  }
  void build() {
    e.build_solve_program();
    e.sync();
    e.factored_ = true;
  }
};

// Both applies are whole once the tree is factored: neither allocates, so a
// full device cannot leave one half built.
void transposed() {
  Made t;
  t.build();
  CHECK(t.e.flow_);
  std::vector<double> b(t.e.nrows_, 1.0);
  fake::dev_limit = 0;
  t.e.perm_.cur_ = t.e.perm_.chunks_.size();  // nothing left in the arenas either
  t.e.flow_mem_.cur_ = t.e.flow_mem_.chunks_.size();
  const long before = fake::n_malloc;
  for (int i = 0; i < 2; ++i) {
    t.e.solve_t_dev(b.data(), b.data());
    t.e.solve_dev(b.data(), b.data());
  }
  CHECK(seen::flow_begins == 4 && seen::flow_parts > 0 && fake::n_malloc == before);
}

// Where the staged program takes over, nothing of the dataflow programs stays.
void staged(Made& t) {
  t.build();
  CHECK(!t.e.flow_ && t.e.flow_mem_.reserved() == 0 && t.e.xbuf_ && t.e.bin_ && !t.e.fwd_.empty());
  for (auto& o : t.e.ops_) CHECK(!o.W);
  for (auto& m : t.e.flow_mode_) CHECK(m.run.empty());
  CHECK(hipGetLastError() == hipSuccess);  // no launch check finds a handled failure
}
void segments() {
  Made t;
  auto& o = t.e.ops_.back();  // one input segment more than the kernel takes
  o.segs.assign(kFlowMaxSegs + 1, {o.c, 1});
  o.m = o.ldv = kFlowMaxSegs + 1;
  o.k = o.kr = 1;
  staged(t);
}
// no memory for the first, or for a later part of a second copy of the reflectors
void no_memory() {
  for (size_t room : {size_t(32) << 20, size_t(96) << 20}) {
    Made t;
    auto o = t.e.ops_[0];
    o.m = o.ldv = 3000;
    o.k = o.kr = o.ldr = 1000;
    for (int i = 0; i < 3; ++i) t.e.ops_.push_back(o);  // 24 MB each
    t.e.scratch_.alloc(1);
    fake::dev_limit = fake::dev_used + room;
    staged(t);
    fake::dev_limit = ~size_t(0);
  }
}

// RRQR rounds after a read-back read the tables of the first ones, also when the
// staging ring was outgrown between two of them and another tree takes what the
// pool has to give.
void rrqr_ring() {
  Engine<double> e(3, 0, 0);
  e.set_tol(1e-2);
  const int k = 20, N = 300, nj = 3;
  std::vector<double> C((size_t)k * N);
  std::vector<Engine<double>::RrqrJob> jobs(nj);
  for (auto& j : jobs) { j.Ct = C.data(); j.k = k; j.N = N; }
  // room for the descriptors, not for the next table
  const size_t room = (sizeof(RrqrDesc<double>) * nj + 255) / 256 * 256;
  std::vector<char> fill(e.stager_.cap_ - e.stager_.off_ - room);
  e.stager_.push_raw(fill.data(), fill.size());
  seen::on_panel = [](const RrqrDesc<double>* d, int nd) {
    for (const long have = fake::n_malloc; fake::n_malloc == have;) {  // all that is pooled
      size_t bytes = 1;
      char* p = pool_take(false, bytes, true);
      std::memset(p, 0xee, bytes);
    }
    CHECK(nd == 3);
    for (int q = 0; q < nd; ++q) {
      CHECK(d[q].k == 20 && d[q].N == 300 && d[q].ldc == 300);
      // the fourth round of two times two ends it
      if (seen::panel_calls == 4) *d[q].st = RrqrState{6, 1, 7, 1, 1.0};
    }
  };
  e.rrqr_blocked(jobs);
  CHECK(seen::panel_calls == 4 && e.stager_.n_grow == 1 && e.stager_.retired_.empty());
  for (auto& j : jobs) CHECK(j.rank == 7);
}

// A wait that timed out is reported once; later applies start without it.
void timeout() {
  Made t;
  t.build();
  std::vector<double> b(t.e.nrows_, 1.0);
  *t.e.solve_err_ = 1;
  bool thrown = false;
  try {
    t.e.check_solve();
  } catch (const Error& e) {
    thrown = e.code == kErrNumeric;
  }
  CHECK(thrown && *t.e.solve_err_ == 0);
  t.e.solve_dev(b.data(), b.data());
  t.e.check_solve();
}

// Memory of closed trees stays for the next ones, and leaves when asked to.
void trim() {
  { Made t; t.build(); }
  const size_t kept = fake::dev_used;
  CHECK(kept > 0 && !fake::pinned.empty());
  const long n = fake::n_malloc;
  { Made t; t.build(); }
  CHECK(fake::n_malloc == n && fake::dev_used == kept);
  Made alive;
  alive.build();
  pool_trim();
  std::vector<double> b(alive.e.nrows_, 1.0);
  alive.e.solve_dev(b.data(), b.data());  // what a tree uses is not pooled
  CHECK(fake::dev_used == kept);
  { Made other; other.build(); }
  CHECK(fake::dev_used > kept);
  pool_trim();
  CHECK(fake::dev_used == kept);
}

// A stream that an error left in a capture does not go to the next tree.
void stream() {
  hipStream_t s;
  { Made t; s = t.e.stream_; }
  { Made t; CHECK(t.e.stream_ == s); fake::capturing.insert(s); }
  CHECK(!fake::streams.count(s));
  Made t;
  CHECK(!fake::capturing.count(t.e.stream_));
}

// The tuner's file, written and read again.
void tuner(const char* path) {
  setenv("SPAQR_TUNE_FILE", path, 1);
  {
    Tuner t;
    t.init("gfx950");
    t.record("slower", 28, {{16, 3.5}, {28, 2.5}}, 1.5);
    t.record("faster", 16, {{16, 0.5}, {28, 2.5}}, 1.5);
    t.record("alone", 40, {{40, 2.0}}, -1);
  }
  Tuner t;
  t.init("gfx950");
  CHECK(t.lookup("slower") == 28 && t.lookup("faster") == 16 && t.lookup("alone") == 40 && t.lookup("none") == -1);
  CHECK(t.prefers_register("slower") == 0 && t.prefers_register("faster") == 1);
  CHECK(t.prefers_register("alone") == -1 && t.prefers_register("none") == -1);
}

// Blocks beyond the kernel's 32-bit byte offsets go to the staged apply: factors,
// and the off-diagonal blocks that the transposed products read.
void offsets() {
  Made t;
  CHECK(t.e.flow_fits());
  auto& o = t.e.ops_.back();
  Engine<double>::Block b{};
  b.ld = 1 << 18;
  o.r12.push_back({b, {o.c, 1 << 10}});
  CHECK(t.e.flow_fits());
  o.r12.back().second.second = 1 << 12;
  CHECK(!t.e.flow_fits());
  o.r12.clear();
  o.ldr = 1 << 30;
  CHECK(!t.e.flow_fits());
}
// What a caller sees when device memory ends: the arenas' code and that of the
// Krylov work space.
void codes() {
  Made t;
  t.build();
  fake::dev_limit = 0;
  auto code = [](auto&& f) {
    try {
      f();
    } catch (const Error& e) {
      return e.code;
    }
    return (int)kOk;
  };
  CHECK(code([&] { t.e.perm_.alloc(size_t(1) << 40); }) == kErrOom);
  CHECK(code([&] { t.e.work_dev(0, size_t(1) << 37); }) == kErrHip);
  fake::dev_limit = ~size_t(0);
  CHECK(code([&] { t.e.work_dev(0, 1000); }) == kOk);  // and the slot is usable again
}
}  // namespace

int main(int argc, char** argv) {
  const std::string c = argc > 1 ? argv[1] : "";
  try {
    if (c == "transposed") transposed();
    else if (c == "segments") segments();
    else if (c == "no_memory") no_memory();
    else if (c == "rrqr_ring") rrqr_ring();
    else if (c == "timeout") timeout();
    else if (c == "trim") trim();
    else if (c == "stream") stream();
    else if (c == "tuner" && argc > 2) tuner(argv[2]);
    else if (c == "offsets") offsets();
    else if (c == "codes") codes();
    else CHECK(!"a known case");
  } catch (const std::exception& e) {
    std::printf("exception: %s\n", e.what());
    return 1;
  }
  std::printf("ok\n");
  std::fflush(stdout);
  std::_Exit(0);  // the host pool's threads sleep
}
