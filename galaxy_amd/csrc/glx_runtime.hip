// Host runtime: device segments, batches and launch sequences.
#include "glx_runtime.h"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <memory>
#include <mutex>
#include <thread>

#include "galaxy_lbvh.h"

namespace glx {

[[noreturn]] void fail(int code, const std::string& msg) { throw Error{code, msg}; }

void check(hipError_t e, const char* what) {
  if (e != hipSuccess)
    fail(e == hipErrorOutOfMemory ? GLX_ENOMEM : GLX_EDEVICE,
         std::string(what) + ": " + hipGetErrorString(e));
}

std::recursive_mutex& device_memory_mutex() {
  static std::recursive_mutex mu;
  return mu;
}

void dev_malloc(void** p, size_t bytes, const char* what) {
  std::lock_guard<std::recursive_mutex> lock(device_memory_mutex());
  *p = nullptr;
  check(hipMalloc(p, bytes), what);
}

void dev_free(void* p) {
  if (!p) return;
  std::lock_guard<std::recursive_mutex> lock(device_memory_mutex());
  (void)hipFree(p);
}

void ensure_device() {
  static std::once_flag once;
  static int status = 0;
  static std::string msg;
  std::call_once(once, [] {
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count <= 0) {
      status = GLX_EDEVICE;
      msg = "no HIP device available";
      return;
    }
    e = hipSetDevice(0);
    if (e != hipSuccess) {
      status = GLX_EDEVICE;
      msg = std::string("hipSetDevice: ") + hipGetErrorString(e);
    }
  });
  if (status) fail(status, msg);
}

// ----------------------------------------------------------------------------------
// Downloads. A copy straight into pageable memory the runtime must first fault in and pin
// page by page (25 MB of positions: 4 ms); and widening after the whole copy leaves the
// link idle. Here pieces of 1 MiB go through pinned buffers, two per lane so that the next
// piece is on the link while the last is written out, and large arrays are written by up to
// four threads, which also share the page faults of a fresh destination. Positions and
// velocities of 2^20 bodies into fresh memory: 7.4 -> 2.8 ms, of 2,000,003: 10.3 -> 4.0 ms.
// The lanes are one pinned block, made once the downloads come to kLaneBytes and given back
// with the last handle: making and freeing it takes about 0.3 ms, which a program that opens a
// handle for one small snapshot would pay in full (two streams per lane and a block each, as
// it was first done: 0.6 ms with one lane, 4.5 with four). Until then, and wherever no lane is
// to be had, the copies are plain ones.
// ----------------------------------------------------------------------------------

namespace {
constexpr size_t kPiece = (size_t)1 << 20;       // bytes on the link per piece
constexpr unsigned kLanes = 8;                   // lanes of the process (16 MiB pinned)
constexpr size_t kPerThread = (size_t)4 << 20;   // device bytes worth another thread
constexpr unsigned kDownloadThreads = 4;
constexpr size_t kLaneBytes = (size_t)4 << 20;

// A lane (two pieces of the block) is used by one thread at a time. The block is portable
// memory: any device's copies may use it.
struct LanePool {
  std::mutex mu;
  std::condition_variable back;
  unsigned char* block = nullptr;
  unsigned taken = 0;              // bit per lane
  size_t plain = 0;                // bytes of plain downloads since a handle was first opened
  size_t users = 0;
};

LanePool& lane_pool() {
  static LanePool* p = new LanePool();  // not destroyed: handles may outlive static objects
  return *p;
}

// Lanes in use at most: GLX_DOWNLOAD_LANES caps them, so that the tests reach the plain
// copies and the waits.
unsigned lane_limit() {
  const char* cap = std::getenv("GLX_DOWNLOAD_LANES");
  const unsigned long v = cap ? std::strtoul(cap, nullptr, 10) : kLanes;
  return v < kLanes ? (unsigned)v : kLanes;
}

// Index of a free lane for a download of `bytes`; with wait, the next to come back if all
// are taken; -1: none.
int lane_take(size_t bytes, bool wait) {
  const unsigned limit = lane_limit();
  if (limit == 0) return -1;
  LanePool& p = lane_pool();
  std::unique_lock<std::mutex> lock(p.mu);
  if (!p.block) {
    if (p.plain + bytes < kLaneBytes) {
      p.plain += bytes;
      return -1;
    }
    std::lock_guard<std::recursive_mutex> device(device_memory_mutex());
    if (hipHostMalloc(reinterpret_cast<void**>(&p.block), kLanes * 2 * kPiece,
                      hipHostMallocPortable) != hipSuccess) {
      (void)hipGetLastError();  // the plain copies take over: nothing for a later call to find
      p.block = nullptr;
      return -1;
    }
  }
  for (;;) {
    for (unsigned k = 0; k < limit; ++k)
      if (!(p.taken >> k & 1u)) {
        p.taken |= 1u << k;
        return (int)k;
      }
    if (!wait) return -1;
    p.back.wait(lock);
  }
}

void lane_give(int k) {
  LanePool& p = lane_pool();
  std::lock_guard<std::mutex> lock(p.mu);
  p.taken &= ~(1u << k);
  p.back.notify_all();  // (a waiter with a lower limit may not be able to use it)
}

void lanes_retain() {
  LanePool& p = lane_pool();
  std::lock_guard<std::mutex> lock(p.mu);
  p.users += 1;
}

void lanes_release() {
  LanePool& p = lane_pool();
  std::lock_guard<std::mutex> lock(p.mu);
  p.users -= 1;
  if (p.users != 0) return;
  p.plain = 0;
  if (!p.block) return;
  std::lock_guard<std::recursive_mutex> device(device_memory_mutex());
  (void)hipHostFree(p.block);
  p.block = nullptr;
}

// One thread's lane during a download. A thread that shares the streams with others waits for
// its copies by events; those belong to the device that is current when the lane is opened,
// which is the streams'.
struct Lane {
  int index = -1;
  unsigned char* buf[2] = {nullptr, nullptr};
  hipEvent_t done[2] = {nullptr, nullptr};

  bool open(size_t bytes, bool wait, bool shared) {
    index = lane_take(bytes, wait);
    if (index < 0) return false;
    for (int k = 0; k < 2; ++k) {
      buf[k] = lane_pool().block + (2 * (size_t)index + k) * kPiece;
      if (shared && hipEventCreateWithFlags(&done[k], hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        done[k] = nullptr;
        close();
        return false;
      }
    }
    return true;
  }
  void close() {
    for (int k = 0; k < 2; ++k)
      if (done[k]) (void)hipEventDestroy(done[k]);
    done[0] = done[1] = nullptr;
    if (index >= 0) lane_give(index);
    index = -1;
  }
};

// Pieces of all arrays, taken in order from `next` by the threads of one download. Their
// copies go to the handle's two streams (one alone: no overlap for a few small pieces).
struct Download {
  const Copyout* outs;
  int n;
  hipStream_t st[2];
  std::atomic<size_t> next{0};
  std::atomic<int> error{hipSuccess};

  static size_t per_piece(const Copyout& o) { return kPiece / (o.widen ? sizeof(float) : sizeof(double)); }
  size_t pieces() const {
    size_t t = 0;
    for (int i = 0; i < n; ++i) t += (outs[i].count + per_piece(outs[i]) - 1) / per_piece(outs[i]);
    return t;
  }
  // Array, first element and count of piece k; false past the end.
  bool piece(size_t k, const Copyout*& o, size_t& first, size_t& count) const {
    for (int i = 0; i < n; ++i) {
      const size_t per = per_piece(outs[i]), c = (outs[i].count + per - 1) / per;
      if (k < c) {
        o = &outs[i];
        first = k * per;
        count = outs[i].count - first < per ? outs[i].count - first : per;
        return true;
      }
      k -= c;
    }
    return false;
  }

  void work(const Lane& lane) {
    struct Held {
      const Copyout* o = nullptr;
      size_t first = 0, count = 0;
    } held[2];
    auto start = [&](int k) {
      Held& h = held[k];
      h.o = nullptr;
      if (error != hipSuccess || !piece(next.fetch_add(1), h.o, h.first, h.count)) {
        h.o = nullptr;
        return;
      }
      const size_t item = h.o->widen ? sizeof(float) : sizeof(double);
      hipError_t r = hipMemcpyAsync(lane.buf[k], static_cast<const char*>(h.o->src) + h.first * item,
                                    h.count * item, hipMemcpyDeviceToHost, st[k]);
      if (r == hipSuccess && lane.done[k]) r = hipEventRecord(lane.done[k], st[k]);
      if (r != hipSuccess) {
        error = r;
        h.o = nullptr;
      }
    };
    start(0);
    for (int k = 0; held[k].o; k ^= 1) {
      start(k ^ 1);
      const hipError_t r =
          lane.done[k] ? hipEventSynchronize(lane.done[k]) : hipStreamSynchronize(st[k]);
      if (r != hipSuccess) {
        error = r;
        break;
      }
      const Held& h = held[k];
      double* dst = h.o->dst + h.first;
      if (h.o->widen) {
        const float* src = reinterpret_cast<const float*>(lane.buf[k]);
        for (size_t q = 0; q < h.count; ++q) dst[q] = (double)src[q];
      } else {
        memcpy(dst, lane.buf[k], h.count * sizeof(double));
      }
    }
    if (error != hipSuccess)  // nothing stays in flight to the lane
      for (int k = 0; k < 2; ++k) (void)hipStreamSynchronize(st[k]);
  }
};

// The same without lanes: whole arrays, f32 through a buffer of their own.
void download_plain(const Copyout* outs, int n, hipStream_t st) {
  std::vector<std::unique_ptr<float[]>> narrow(n);
  for (int i = 0; i < n; ++i)
    if (outs[i].widen) narrow[i].reset(new float[outs[i].count]);
  hipError_t r = hipSuccess;
  for (int i = 0; i < n && r == hipSuccess; ++i) {
    const Copyout& o = outs[i];
    r = hipMemcpyAsync(o.widen ? (void*)narrow[i].get() : (void*)o.dst, o.src,
                       o.count * (o.widen ? sizeof(float) : sizeof(double)), hipMemcpyDeviceToHost,
                       st);
  }
  const hipError_t w = hipStreamSynchronize(st);
  check(r != hipSuccess ? r : w, "download");
  for (int i = 0; i < n; ++i)
    if (outs[i].widen)
      for (size_t q = 0; q < outs[i].count; ++q) outs[i].dst[q] = (double)narrow[i][q];
}

// Makes a device current for a scope.
struct OnDevice {
  int was = -1;
  explicit OnDevice(int device) {
    int now = 0;
    check(hipGetDevice(&now), "hipGetDevice");
    if (now == device) return;
    check(hipSetDevice(device), "hipSetDevice");
    was = now;
  }
  ~OnDevice() {
    if (was >= 0) (void)hipSetDevice(was);
  }
};
}  // namespace

void download(const Copyout* outs, int n, const Batch& batch) {
  const hipStream_t st = batch.stream();
  check(hipStreamSynchronize(st), "hipStreamSynchronize");
  Download d{outs, n, {st, batch.side()}};
  size_t bytes = 0;
  for (int i = 0; i < n; ++i) bytes += outs[i].count * (outs[i].widen ? sizeof(float) : sizeof(double));
  if (bytes == 0) return;
  hipDevice_t device = 0;  // the handle's, whatever is current in this thread; new threads start at 0
  check(hipStreamGetDevice(st, &device), "hipStreamGetDevice");
  OnDevice on(device);
  size_t threads = bytes / kPerThread;
  const size_t pieces = d.pieces();
  if (threads > pieces) threads = pieces;
  if (threads > kDownloadThreads) threads = kDownloadThreads;
  Lane mine;
  if (!mine.open(bytes, true, threads > 1)) return download_plain(outs, n, st);
  std::thread more[kDownloadThreads];
  size_t started = 0;
  for (size_t t = 1; t < threads; ++t) {
    try {
      more[started] = std::thread([&d, bytes, device] {
        Lane lane;
        if (hipSetDevice(device) != hipSuccess || !lane.open(bytes, false, true))
          return;  // the others take its pieces
        d.work(lane);
        lane.close();
      });
    } catch (...) {
      break;  // no thread to be had: the same
    }
    ++started;
  }
  d.work(mine);
  for (size_t t = 0; t < started; ++t) more[t].join();
  mine.close();
  check((hipError_t)d.error.load(), "download");
}

static inline size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// ----------------------------------------------------------------------------------
// Segment
// ----------------------------------------------------------------------------------

namespace {
struct Carve {
  size_t off = 0;
  template <class T>
  size_t take(size_t count) {
    const size_t o = off;
    off = align_up(off + count * sizeof(T), 256);
    return o;
  }
};

struct Layout {
  size_t x, v, m, acc, acc_out, k0, k1, v0, v1, leaf, node, box, quad, topo, pleaf, flag,
      strad, strad2, scount, scount2, scount3, gend, bbox, bounds, counters, total;
};

Layout layout_for(uint32_t n, bool with_acc_out) {
  const size_t N = n ? n : 1;
  Carve c;
  Layout L;
  L.x = c.take<double>(3 * N);
  L.v = c.take<float>(3 * N);
  L.m = c.take<double>(N);
  L.acc = c.take<float>(3 * N);
  L.acc_out = with_acc_out ? c.take<double>(3 * N) : 0;
  L.k0 = c.take<uint64_t>(N);
  L.k1 = c.take<uint64_t>(N);
  L.v0 = c.take<uint32_t>(N);
  L.v1 = c.take<uint32_t>(N);
  // leaves, classifier records and quadrupoles adjacent: the group walk addresses all
  // three with 32-bit byte offsets from the leaf array (80 B per body)
  L.leaf = c.take<float4>(N);
  L.node = c.take<Node>(N);
  L.quad = c.take<float4>(2 * N);
  L.box = c.take<NodeBox>(N);
  L.topo = c.take<uint4>(N);
  L.pleaf = c.take<uint32_t>(N);
  L.flag = c.take<uint32_t>(N);
  L.strad = c.take<uint32_t>(N);
  L.strad2 = c.take<uint32_t>(N);
  L.scount = c.take<uint32_t>((N + kAggTile - 1) / kAggTile);
  L.scount2 = c.take<uint32_t>((N + kMidSpan - 1) / kMidSpan);
  L.scount3 = c.take<uint32_t>((N + kMid2Span - 1) / kMid2Span);
  L.gend = c.take<uint32_t>(N);
  L.bbox = c.take<unsigned long long>(6);
  L.bounds = c.take<double>(8);
  L.counters = c.take<unsigned long long>(kCounters);
  L.total = c.off;
  return L;
}
}  // namespace

size_t Segment::bytes_for(uint32_t n, bool with_acc_out) {
  return layout_for(n, with_acc_out).total;
}

Segment::~Segment() { dev_free(block_); }

void Segment::reserve(uint32_t n, bool with_acc_out) {
  if (block_ && n <= capacity && (has_acc_out || !with_acc_out)) return;
  uint32_t cap = n;
  if (block_ && n > capacity) cap = n > capacity + capacity / 2 ? n : capacity + capacity / 2;
  const bool acc_out = with_acc_out || has_acc_out;
  const Layout L = layout_for(cap, acc_out);
  std::lock_guard<std::recursive_mutex> lock(device_memory_mutex());
  void* blk = nullptr;
  dev_malloc(&blk, L.total, "hipMalloc(segment)");
  // arrival flags and counters must start at zero (kernels keep them zero afterwards)
  hipError_t e = hipMemset(static_cast<char*>(blk) + L.flag, 0, sizeof(uint32_t) * (cap ? cap : 1));
  if (e == hipSuccess)
    e = hipMemset(static_cast<char*>(blk) + L.counters, 0, kCounters * sizeof(unsigned long long));
  if (e != hipSuccess) {
    dev_free(blk);
    check(e, "hipMemset(segment)");
  }
  dev_free(block_);
  block_ = blk;
  bytes_ = L.total;
  capacity = cap;
  has_acc_out = acc_out;
  char* b = static_cast<char*>(blk);
  SegDesc d = desc;
  d.x = reinterpret_cast<double*>(b + L.x);
  d.v = reinterpret_cast<float*>(b + L.v);
  d.m = reinterpret_cast<double*>(b + L.m);
  d.acc = reinterpret_cast<float*>(b + L.acc);
  d.acc_out = acc_out ? reinterpret_cast<double*>(b + L.acc_out) : nullptr;
  d.keys[0] = b + L.k0;
  d.keys[1] = b + L.k1;
  d.vals[0] = reinterpret_cast<uint32_t*>(b + L.v0);
  d.vals[1] = reinterpret_cast<uint32_t*>(b + L.v1);
  d.leaf = reinterpret_cast<float4*>(b + L.leaf);
  d.node = reinterpret_cast<Node*>(b + L.node);
  d.box = reinterpret_cast<NodeBox*>(b + L.box);
  d.quad = reinterpret_cast<float4*>(b + L.quad);
  d.topo = reinterpret_cast<uint4*>(b + L.topo);
  d.parent_leaf = reinterpret_cast<uint32_t*>(b + L.pleaf);
  d.flag = reinterpret_cast<uint32_t*>(b + L.flag);
  d.strad = reinterpret_cast<uint32_t*>(b + L.strad);
  d.strad2 = reinterpret_cast<uint32_t*>(b + L.strad2);
  d.scount = reinterpret_cast<uint32_t*>(b + L.scount);
  d.scount2 = reinterpret_cast<uint32_t*>(b + L.scount2);
  d.scount3 = reinterpret_cast<uint32_t*>(b + L.scount3);
  d.gend = reinterpret_cast<uint32_t*>(b + L.gend);
  d.bbox = reinterpret_cast<unsigned long long*>(b + L.bbox);
  d.bounds = reinterpret_cast<double*>(b + L.bounds);
  d.counters = reinterpret_cast<unsigned long long*>(b + L.counters);
  desc = d;
}

// ----------------------------------------------------------------------------------
// Batch
// ----------------------------------------------------------------------------------

// The side stream and its events exist from construction, so that a step graph captured
// on the batch stream never creates them mid-capture.
Batch::Batch(hipStream_t st) : stream_(st) {
  check(hipStreamCreateWithFlags(&side_, hipStreamNonBlocking), "hipStreamCreate");
  if (hipEventCreateWithFlags(&fork_, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&join_, hipEventDisableTiming) != hipSuccess) {
    if (fork_) (void)hipEventDestroy(fork_);
    (void)hipStreamDestroy(side_);
    fail(GLX_EDEVICE, "hipEventCreate failed");
  }
  lanes_retain();
}

Batch::~Batch() {
  lanes_release();
  if (fork_) (void)hipEventDestroy(fork_);
  if (join_) (void)hipEventDestroy(join_);
  if (side_) (void)hipStreamDestroy(side_);
  dev_free(segs_);
  dev_free(etiles_);
  dev_free(atiles_);
  dev_free(mtiles_);
  dev_free(m2tiles_);
  dev_free(ctiles_);
  dev_free(chunk_rows_);
  dev_free(btiles_);
  dev_free(split_key_);
  dev_free(wtiles_);
  dev_free(gtiles_);
  dev_free(tile_hist_);
  dev_free(diag_partial_);
  dev_free(diag_out_);
}

template <class T>
static void grow(T*& p, size_t& cap, size_t need) {
  if (need <= cap && p) return;
  size_t c = need > cap * 2 ? need : cap * 2;
  if (c == 0) c = 1;
  T* q = nullptr;
  dev_malloc(reinterpret_cast<void**>(&q), c * sizeof(T), "hipMalloc(batch table)");
  dev_free(p);
  p = q;
  cap = c;
}

static void push_tiles(std::vector<Tile>& v, uint32_t seg, uint32_t n, uint32_t size) {
  for (uint32_t st = 0; st < n; st += size)
    v.push_back(Tile{seg, st, (n - st) < size ? n - st : size, 0});
}

void Batch::set_segments(const std::vector<SegDesc>& descs) {
  host_ = descs;
  nseg_ = (uint32_t)descs.size();
  std::vector<Tile> et, at, mt, m2, ct, wt, gt, bt;
  uint64_t total = 0;
  uint32_t largest = 0;
  split_ = false;
  multi_tile_ = false;
  chunked_ = false;
  // GLX_WALK_WIDE=1 takes the 64-bit-address walk for every segment (the two forms give
  // the same results bit for bit; the tests compare them on systems of any size)
  const char* force_wide = std::getenv("GLX_WALK_WIDE");
  wide_ = force_wide && force_wide[0] == '1';
  // GLX_WALK_STACK_CAP=k caps the group walk's stack at k entries, so that the tests can
  // drive groups into the per-target fallback (default: the full LDS stack)
  const char* cap = std::getenv("GLX_WALK_STACK_CAP");
  const uint32_t stack_cap = cap ? (uint32_t)std::strtoul(cap, nullptr, 10) : 0u;
  for (uint32_t s = 0; s < nseg_; ++s) {
    SegDesc& d = host_[s];
    d.stack_cap = stack_cap;
    if (!walk_off32((uint64_t)d.leaf, (uint64_t)d.node, (uint64_t)d.quad, d.n)) wide_ = true;
    d.sort_tile0 = (uint32_t)et.size();
    push_tiles(et, s, d.n, kSortTile);
    d.sort_tiles = (uint32_t)et.size() - d.sort_tile0;
    d.scan_chunk0 = (uint32_t)ct.size();
    d.scan_len = (d.sort_tiles + kScanRows - 1) / kScanRows;
    if (d.scan_len < kScanChunk) d.scan_len = kScanChunk;
    for (uint32_t c = 0; c < d.sort_tiles; c += d.scan_len)
      ct.push_back(Tile{s, d.sort_tile0 + c, std::min(d.sort_tiles - c, d.scan_len),
                        d.sort_tiles <= d.scan_len ? 1u : 0u});
    d.scan_chunks = (uint32_t)ct.size() - d.scan_chunk0;
    if (d.scan_chunks > 1) chunked_ = true;
    push_tiles(at, s, d.n, kAggTile);
    total += d.n;
    if (d.n > largest) largest = d.n;
    if (d.n > (uint32_t)kAggTile) multi_tile_ = true;
    if (d.n > kMidMin) push_tiles(mt, s, d.n, kMidSpan);
    if (d.n > kMid2Min) push_tiles(m2, s, d.n, kMid2Span);
    push_tiles(wt, s, d.n, kBlock);
    push_tiles(gt, s, d.n, kGroup);
  }
  if (largest <= kLocalMax && total <= kLocalTotal)
    for (uint32_t s = 0; s < nseg_; ++s) {
      const uint32_t n = host_[s].n, nb = n ? local_buckets(n) : 0u;
      for (uint32_t b = 0; b < nb; ++b) bt.push_back(Tile{s, b, 0u, nb > 1u ? 1u : 0u});
      if (nb > 1u) split_ = true;
    }
  n_bt_ = (uint32_t)bt.size();
  n_et_ = (uint32_t)et.size();
  n_at_ = (uint32_t)at.size();
  n_mt_ = (uint32_t)mt.size();
  n_m2_ = (uint32_t)m2.size();
  n_ct_ = (uint32_t)ct.size();
  n_wt_ = (uint32_t)wt.size();
  n_gt_ = (uint32_t)gt.size();
  size_t cs = cap_segs_;
  grow(segs_, cs, nseg_ ? nseg_ : 1);
  if (cs != cap_segs_ || !diag_out_) {
    dev_free(diag_out_);
    diag_out_ = nullptr;
    dev_malloc(reinterpret_cast<void**>(&diag_out_), cs * kDiagRecord * sizeof(double),
               "hipMalloc(diag)");
  }
  if (split_ && (cs != split_segs_ || !split_key_)) {
    dev_free(split_key_);
    split_key_ = nullptr;
    split_segs_ = 0;
    const size_t words = 2 * kSplitMax + kSplitMax + kSplitMax + 1;  // u64 keys, indices, starts
    dev_malloc(reinterpret_cast<void**>(&split_key_), cs * words * sizeof(uint32_t) + 8,
               "hipMalloc(splitters)");
    split_segs_ = cs;
  }
  cap_segs_ = cs;
  size_t ce = cap_et_;
  grow(etiles_, ce, n_et_ ? n_et_ : 1);
  if (ce != cap_et_ || !tile_hist_) {
    dev_free(tile_hist_);
    dev_free(diag_partial_);
    tile_hist_ = nullptr;
    diag_partial_ = nullptr;
    dev_malloc(reinterpret_cast<void**>(&tile_hist_), ce * kRadixBinsMax * sizeof(uint32_t),
               "hipMalloc(hist)");
    dev_malloc(reinterpret_cast<void**>(&diag_partial_), ce * kDiagRecord * sizeof(double),
               "hipMalloc(diag)");
  }
  cap_et_ = ce;
  grow(atiles_, cap_at_, n_at_ ? n_at_ : 1);
  grow(mtiles_, cap_mt_, n_mt_ ? n_mt_ : 1);
  grow(m2tiles_, cap_m2_, n_m2_ ? n_m2_ : 1);
  size_t cc = cap_ct_;
  grow(ctiles_, cc, n_ct_ ? n_ct_ : 1);
  if (cc != cap_ct_ || !chunk_rows_) {
    dev_free(chunk_rows_);
    chunk_rows_ = nullptr;
    dev_malloc(reinterpret_cast<void**>(&chunk_rows_), cc * kRadixBinsMax * sizeof(uint32_t),
               "hipMalloc(scan chunks)");
  }
  cap_ct_ = cc;
  grow(btiles_, cap_bt_, n_bt_ ? n_bt_ : 1);
  grow(wtiles_, cap_wt_, n_wt_ ? n_wt_ : 1);
  grow(gtiles_, cap_gt_, n_gt_ ? n_gt_ : 1);
  auto up = [&](void* dst, const void* src, size_t bytes) {
    if (bytes)
      check(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream_), "upload table");
  };
  up(segs_, host_.data(), nseg_ * sizeof(SegDesc));
  up(etiles_, et.data(), n_et_ * sizeof(Tile));
  up(atiles_, at.data(), n_at_ * sizeof(Tile));
  up(mtiles_, mt.data(), n_mt_ * sizeof(Tile));
  up(m2tiles_, m2.data(), n_m2_ * sizeof(Tile));
  up(ctiles_, ct.data(), n_ct_ * sizeof(Tile));
  up(btiles_, bt.data(), n_bt_ * sizeof(Tile));
  up(wtiles_, wt.data(), n_wt_ * sizeof(Tile));
  up(gtiles_, gt.data(), n_gt_ * sizeof(Tile));
  check(hipStreamSynchronize(stream_), "set_segments");
}

void Batch::set_dt(double dt) {
  for (auto& d : host_) {
    d.dt = dt;
    d.half_dt = (float)(0.5 * dt);
  }
  if (nseg_)
    check(hipMemcpyAsync(segs_, host_.data(), nseg_ * sizeof(SegDesc), hipMemcpyHostToDevice,
                         stream_),
          "upload segments");
  check(hipStreamSynchronize(stream_), "set_dt");
}

void Batch::set_active(const uint8_t* mask) {
  bool same = true;
  for (auto& d : host_) {
    same = same && d.active == mask;
    d.active = mask;
  }
  if (same) return;
  if (nseg_)
    check(hipMemcpyAsync(segs_, host_.data(), nseg_ * sizeof(SegDesc), hipMemcpyHostToDevice,
                         stream_),
          "upload segments");
  check(hipStreamSynchronize(stream_), "set_active");
}

void Batch::reset_bbox() { check(launch_seg_reset(stream_, segs_, nseg_), "seg_reset"); }
void Batch::bbox() { check(launch_bbox(stream_, segs_, etiles_, n_et_), "bbox"); }
void Batch::kick_drift_bbox() {
  check(launch_kick_drift_bbox(stream_, segs_, etiles_, n_et_), "kick_drift");
}
void Batch::encode(uint32_t* lanes_out) {
  check(launch_encode(stream_, mode_, segs_, etiles_, n_et_, lanes_out), "encode");
}
void Batch::bounds_only() { check(launch_bounds_only(stream_, mode_, segs_, nseg_), "bounds"); }
void Batch::iota() { check(launch_iota(stream_, mode_, segs_, etiles_, n_et_), "iota"); }
void Batch::sort() {
  uint32_t* idx = reinterpret_cast<uint32_t*>(split_key_ + split_segs_ * kSplitMax);
  const SplitTable table{split_key_, idx, idx + split_segs_ * kSplitMax};
  const SortScratch sc{tile_hist_, ctiles_, n_ct_, chunk_rows_, chunked_,
                       btiles_,    n_bt_,   split_, table};
  check(launch_sort(stream_, mode_, segs_, nseg_, etiles_, n_et_, sc), "sort");
}
void Batch::gather() { check(launch_gather(stream_, segs_, etiles_, n_et_), "gather"); }
void Batch::refresh_leaves() {
  check(launch_refresh_leaves(stream_, segs_, etiles_, n_et_), "refresh leaves");
}
void Batch::karras() { check(launch_karras(stream_, mode_, segs_, etiles_, n_et_), "karras"); }
void Batch::aggregate() {
  const AggTiles t{atiles_, mtiles_, m2tiles_, n_at_, n_mt_, n_m2_, multi_tile_};
  check(launch_aggregate(stream_, mode_, segs_, nseg_, t), "aggregate");
}
void Batch::flatten(const FlatOut& out) {
  check(launch_flatten(stream_, segs_, etiles_, n_et_, out), "flatten");
}
void Batch::walk(int mode, bool count) {
  check(launch_walk(stream_, mode_, segs_, wtiles_, n_wt_, gtiles_, n_gt_, mode, count, wide_),
        "walk");
}

void Batch::build_and_walk(int mode, bool count) {
  encode();
  sort();
  // the gather (HBM-bound) beside the tree build (latency-bound): both read only the
  // sort's output and write disjoint arrays; the bottom-up pass needs both
  check(hipEventRecord(fork_, stream_), "hipEventRecord");
  check(hipStreamWaitEvent(side_, fork_, 0), "hipStreamWaitEvent");
  check(launch_gather(side_, segs_, etiles_, n_et_), "gather");
  check(hipEventRecord(join_, side_), "hipEventRecord");
  karras();
  check(hipStreamWaitEvent(stream_, join_, 0), "hipStreamWaitEvent");
  aggregate();
  walk(mode, count);
}

void Batch::diag(double* host_out) {
  check(launch_diag(stream_, segs_, nseg_, etiles_, n_et_, diag_partial_, diag_out_), "diag");
  check(hipMemcpyAsync(host_out, diag_out_, nseg_ * kDiagRecord * sizeof(double),
                       hipMemcpyDeviceToHost, stream_), "diag download");
  check(hipStreamSynchronize(stream_), "diag");
}

}  // namespace glx
