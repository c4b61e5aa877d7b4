#include "common.hpp"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

namespace spq {

std::recursive_mutex& capture_lock() {
  static std::recursive_mutex m;
  return m;
}

long Arena::n_chunks = 0;
double Arena::t_chunks = 0;

void* Arena::alloc(size_t bytes, size_t align) {
  if (bytes == 0) bytes = align;
  while (cur_ < chunks_.size()) {
    Chunk& c = chunks_[cur_];
    size_t off = (c.off + align - 1) / align * align;
    if (off + bytes <= c.size) {
      c.off = off + bytes;
      used_ += bytes;
      return c.p + off;
    }
    ++cur_;
  }
  size_t sz = bytes > chunk_ ? (bytes + align) : chunk_;
  const double t0 = wall();
  if (chunks_.empty()) SPQ_HIP(hipGetDevice(&dev_));
  char* p = nullptr;
  try {
    p = pool_take(false, sz);
  } catch (const Error& e) {
    throw Error(kErrOom, "device allocation of " + std::to_string(sz) + " bytes failed: " + e.what());
  }
  t_chunks += wall() - t0;
  ++n_chunks;
  chunks_.push_back({p, sz, 0});
  reserved_ += sz;
  cur_ = chunks_.size() - 1;
  Chunk& c = chunks_.back();
  c.off = bytes;
  used_ += bytes;
  return c.p;
}

void Arena::rewind() {
  for (auto& c : chunks_) c.off = 0;
  cur_ = 0;
  used_ = 0;
}

void Arena::release() {
  for (auto& c : chunks_) pool_give(false, c.p, c.size, dev_);
  chunks_.clear();
  cur_ = 0;
  used_ = 0;
  reserved_ = 0;
}

namespace {
struct PoolEntry { int dev; bool host; size_t bytes; char* p; };
// kept per device: device memory (the arenas of a tree of a million unknowns; 3%
// of the device's), and pinned host memory
constexpr size_t kPoolBytes[2] = {size_t(8) << 30, size_t(2) << 30};
constexpr size_t kPoolStreams = 16;
std::mutex& pool_mu() {
  static std::mutex m;
  return m;
}
// never destroyed: buffers still pooled at exit are left to the process end
// (freeing them would race the HIP runtime's own teardown)
std::vector<PoolEntry>& pool() {
  static std::vector<PoolEntry>* v = new std::vector<PoolEntry>();
  return *v;
}
}  // namespace

char* pool_take(bool host, size_t& bytes, bool largest) {
  int dev = 0;
  SPQ_HIP(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lk(pool_mu());
    auto& v = pool();
    int best = -1;
    for (size_t i = 0; i < v.size(); ++i)
      if (v[i].dev == dev && v[i].host == host && v[i].bytes >= bytes &&
          (largest || v[i].bytes <= 2 * bytes + (size_t(1) << 20)) &&  // no large chunk for a small request
          (best < 0 || (largest ? v[i].bytes > v[best].bytes : v[i].bytes < v[best].bytes)))
        best = (int)i;
    if (best >= 0) {
      char* p = v[best].p;
      bytes = v[best].bytes;
      v.erase(v.begin() + best);
      return p;
    }
  }
  void* p = nullptr;
  if (host) SPQ_HIP(host_malloc(&p, bytes));
  else SPQ_HIP(dev_malloc(&p, bytes));
  return (char*)p;
}

// Device memory; when there is none left, what the pool keeps is given back
// and the allocation tried again.
hipError_t dev_malloc(void** p, size_t bytes) {
  std::lock_guard<std::recursive_mutex> lk(capture_lock());
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return e;
  std::vector<PoolEntry> drop;
  {
    std::lock_guard<std::mutex> lk2(pool_mu());
    auto& v = pool();
    for (size_t i = 0; i < v.size();)
      if (v[i].dev == dev && !v[i].host) {
        drop.push_back(v[i]);
        v.erase(v.begin() + i);
      } else {
        ++i;
      }
  }
  if (drop.empty()) return e;
  (void)hipGetLastError();
  for (auto& d : drop) (void)hipFree(d.p);
  return hipMalloc(p, bytes);
}

void pool_trim() {
  std::vector<PoolEntry> drop;
  {
    std::lock_guard<std::mutex> lk(pool_mu());
    drop.swap(pool());
  }
  for (auto& e : drop) {
    if (e.host) host_free(e.p);
    else dev_free(e.p);
  }
}

namespace {
std::vector<std::pair<int, hipStream_t>>& stream_pool() {
  static auto* v = new std::vector<std::pair<int, hipStream_t>>();
  return *v;
}
}  // namespace

hipStream_t stream_take() {
  int dev = 0;
  SPQ_HIP(hipGetDevice(&dev));
  {
    std::lock_guard<std::mutex> lk(pool_mu());
    auto& v = stream_pool();
    for (size_t i = 0; i < v.size(); ++i)
      if (v[i].first == dev) {
        const hipStream_t s = v[i].second;
        v.erase(v.begin() + i);
        return s;
      }
  }
  hipStream_t s = nullptr;
  SPQ_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  return s;
}

void stream_give(hipStream_t s, int dev) {
  if (!s) return;
  // a capture that an error left open, or an error on the stream, must not
  // reach the next tree
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  const bool idle = hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone &&
                    hipStreamSynchronize(s) == hipSuccess;
  if (idle) {
    std::lock_guard<std::mutex> lk(pool_mu());
    auto& v = stream_pool();
    size_t n = 0;
    for (auto& e : v) n += e.first == dev;
    if (n < kPoolStreams) {
      v.push_back({dev, s});
      return;
    }
  }
  std::lock_guard<std::recursive_mutex> lk(capture_lock());
  (void)hipStreamDestroy(s);
}

void pool_give(bool host, char* p, size_t bytes, int dev) {
  if (!p) return;
  std::vector<PoolEntry> drop;
  {
    std::lock_guard<std::mutex> lk(pool_mu());
    auto& v = pool();
    v.push_back({dev, host, bytes, p});
    // over the limit: free the smallest buffers of this kind and device
    for (;;) {
      size_t tot = 0;
      int small = -1;
      for (size_t i = 0; i < v.size(); ++i) {
        if (v[i].dev != dev || v[i].host != host) continue;
        tot += v[i].bytes;
        if (small < 0 || v[i].bytes < v[small].bytes) small = (int)i;
      }
      if (tot <= kPoolBytes[host] || small < 0) break;
      drop.push_back(v[small]);
      v.erase(v.begin() + small);
    }
  }
  for (auto& e : drop) {
    if (e.host) host_free(e.p);
    else dev_free(e.p);
  }
}

Stager::~Stager() {
  release_retired();
  pool_give(true, host_, host_bytes_, device_);
  pool_give(false, dev_, dev_bytes_, device_);
  if (up_host_) pool_give(true, up_host_, up_cap_, device_);
}

void Stager::release_retired() {
  for (auto& r : retired_) {
    pool_give(true, r.host, r.host_bytes, device_);
    pool_give(false, r.dev, r.dev_bytes, device_);
  }
  retired_.clear();
}

void Stager::upload_raw(void* dst, const void* src, size_t bytes) {
  constexpr size_t kUpCap = size_t(32) << 20;
  if (!up_host_) {
    up_cap_ = kUpCap;
    up_host_ = pool_take(true, up_cap_);
    up_off_ = 0;
  }
  if (bytes > up_cap_) {  // larger than the buffer: a synchronous copy
    flush_uploads();
    SPQ_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream_));
    SPQ_HIP(hipStreamSynchronize(stream_));
    return;
  }
  if (up_off_ + bytes > up_cap_) {  // every earlier upload must have landed
    flush_uploads();
    SPQ_HIP(hipStreamSynchronize(stream_));
    up_off_ = 0;
  }
  std::memcpy(up_host_ + up_off_, src, bytes);
  char* d = (char*)dst;
  // the pending copy grows when this table sits at the same distance from
  // its start on the device as in the staging buffer (the bytes in between
  // are alignment padding of the earlier destination)
  if (up_pend_bytes_ && d == up_pend_dev_ + (up_off_ - up_pend_host_)) {
    up_pend_bytes_ = up_off_ - up_pend_host_ + bytes;
  } else {
    flush_uploads();
    up_pend_host_ = up_off_;
    up_pend_dev_ = d;
    up_pend_bytes_ = bytes;
  }
  up_off_ += (bytes + 255) / 256 * 256;
}

void Stager::flush_uploads() {
  if (!up_pend_bytes_) return;
  SPQ_HIP(hipMemcpyAsync(up_pend_dev_, up_host_ + up_pend_host_, up_pend_bytes_, hipMemcpyHostToDevice, stream_));
  up_pend_bytes_ = 0;
}

void Stager::init(hipStream_t s, size_t bytes) {
  stream_ = s;
  SPQ_HIP(hipGetDevice(&device_));
  host_bytes_ = bytes;
  host_ = pool_take(true, host_bytes_, true);  // a ring an earlier tree grew
  dev_bytes_ = host_bytes_;
  dev_ = pool_take(false, dev_bytes_);
  cap_ = host_bytes_;
  off_ = 0;
}

const void* Stager::push_raw(const void* src, size_t bytes) {
  if (bytes == 0) return nullptr;
  size_t need = (bytes + 255) / 256 * 256;
  if (off_ + need > cap_ && cap_ < kMaxRing) {
    // grow: what is pending is copied from the old ring, which stays with
    // its readers until the next synchronisation.  Without memory for a
    // larger ring the old one wraps below.
    size_t want = cap_;
    while (want < kMaxRing && want < need) want *= 2;
    if (want < kMaxRing) want *= 2;
    want = std::max(std::min(want, kMaxRing), need);
    size_t hb = want, db = 0;
    char *nh = nullptr, *nd = nullptr;
    try {
      nh = pool_take(true, hb);
      db = hb;
      nd = pool_take(false, db);
    } catch (const Error&) {
      (void)hipGetLastError();
      if (nh) pool_give(true, nh, hb, device_);
      nh = nd = nullptr;
    }
    if (nh && nd) {
      flush();
      retired_.push_back({host_, dev_, host_bytes_, dev_bytes_});
      host_ = nh; host_bytes_ = hb;
      dev_ = nd; dev_bytes_ = db;
      cap_ = hb;
      off_ = 0;
      pend_ = 0;
      ++n_grow;
    }
  }
  if (need > cap_) throw Error(kErrOom, "descriptor table larger than the staging ring");
  if (off_ + need > cap_) {
    // wrap: copy what is pending, let every reader of the ring finish
    flush();
    SPQ_HIP(hipStreamSynchronize(stream_));
    off_ = 0;
    pend_ = 0;
    release_retired();
    ++n_wrap;
  }
  std::memcpy(host_ + off_, src, bytes);
  const void* d = dev_ + off_;
  off_ += need;
  return d;
}

void Stager::flush() {
  flush_uploads();
  if (off_ > pend_) SPQ_HIP(hipMemcpyAsync(dev_ + pend_, host_ + pend_, off_ - pend_, hipMemcpyHostToDevice, stream_));
  pend_ = off_;
}

}  // namespace spq
