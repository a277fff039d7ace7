// HIP kernels of the simplifier for CDNA4 (gfx950, wave64).
//
// Work mapping:
//   * clause-parallel stages (BCP clean-up, counting, compaction) use one
//     thread per clause;
//   * the occurrence table is built by literal ranges: 1024-thread
//     workgroups per tile of clauses count and partition the occurrences
//     by range in LDS (in two steps for many literals), then one workgroup
//     per range counts, scans and places its lists in LDS (no global atomic
//     per occurrence); one workgroup does it all for small formulas;
//   * list-parallel stages (BCP visits, list deletions) use one workgroup
//     per occurrence list with the threads striding the list; narrow levels
//     of root propagation share one launch of one workgroup;
//   * SUB and BVE use groups of 2 to 64 lanes per elected variable on a copy
//     of its lists in LDS, the LCVE election 1 to 16 lanes per candidate on
//     the pool, BCE and ERE a thread per variable or pair;
//   * scans and the stable radix sort use 256-thread workgroups with
//     wave64 shuffles for the in-wave prefix and LDS for the wave totals,
//     short ones one workgroup of 1,024.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <thread>
#include <vector>
#include <stdexcept>
#include <string>

#include "pfs_launch.hpp"
#include "pfs_staging.hpp"

namespace pfs {

#define PFS_HIP(call)                                                                      \
  do {                                                                                     \
    hipError_t e_ = (call);                                                                \
    if (e_ != hipSuccess)                                                                  \
      throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e_) + " at " + \
                               __FILE__ + ":" + std::to_string(__LINE__));                 \
  } while (0)

struct KRec {
  const char* name;
  hipEvent_t a, b;
};
// Small device-to-host reads (counts, flags, a few records) land in pinned
// staging memory: a copy into pageable memory makes the runtime stage it
// itself, which adds tens of microseconds to every read-and-wait.  The
// copies to their destinations happen in stream_sync, which every caller
// runs before it looks at what it read.
constexpr size_t PIN_BYTES = 64 << 10, PIN_SMALL = 4096;
struct PinCopy {
  void* dst;
  size_t off, bytes;
};
// The smallest reads (a few counters before every wait) are gathered and
// written to the pinned area by one kernel launched when the caller waits,
// with a flag behind them that the waiting thread polls: a counter read
// takes 9.9 us after its kernel that way, 14.3 with a copy and a wait for the
// stream (a small formula's round waits eight times).  Anything else put on
// the stream before the wait launches the gathered reads first, so a read
// sees what the stream held when it was asked for.
constexpr u32 PUB_MAX = 6, PUB_BYTES = 256;
struct PubSet {
  const u32* src[PUB_MAX];
  u32* dst[PUB_MAX];
  u32 words[PUB_MAX];
};
struct Stream {
  hipStream_t s;
  int device;
  bool prof = false;        // record events around every kernel launch
  std::vector<KRec> recs;   // pending event pairs
  unsigned char* pin = nullptr;  // PIN_BYTES of pinned host memory
  size_t pin_used = 0;
  std::vector<PinCopy> pend;     // staged reads not yet copied out
  PubSet pub = {};               // gathered reads, not launched yet
  u32 npub = 0;
  u32* flag = nullptr;           // in the pinned area, past PIN_BYTES
  u32 tag = 0;                   // its value once the last gathered reads have landed
};
static void pub_flush(Stream* st, bool flagged);
// before anything is put on the stream
static inline void stream_op(Stream* st) {
  if (st->npub) pub_flush(st, false);
}
static void pin_flush(Stream* st) {
  for (const PinCopy& c : st->pend) memcpy(c.dst, st->pin + c.off, c.bytes);
  st->pend.clear();
  st->pin_used = 0;
}
struct Event {
  hipEvent_t e;
};

static inline unsigned grid_for(size_t n, unsigned block) {
  return (unsigned)((n + block - 1) / block);
}
#define LAUNCH_CHECK() PFS_HIP(hipGetLastError())
// launch on the context stream; with profiling on, bracket it with events
#define KLAUNCH(kern, grid, block, st, ...) KLAUNCH_LDS(kern, grid, block, 0, st, __VA_ARGS__)
// the same with 'lds' bytes of dynamic LDS reserved per workgroup
#define KLAUNCH_LDS(kern, grid, block, lds, st, ...)          \
  do {                                                         \
    stream_op(st);                                             \
    hipEvent_t e0_ = nullptr;                                  \
    if ((st)->prof) {                                          \
      PFS_HIP(hipEventCreate(&e0_));                           \
      PFS_HIP(hipEventRecord(e0_, (st)->s));                   \
    }                                                          \
    kern<<<(grid), (block), (lds), (st)->s>>>(__VA_ARGS__);    \
    LAUNCH_CHECK();                                            \
    if ((st)->prof) {                                          \
      hipEvent_t e1_;                                          \
      PFS_HIP(hipEventCreate(&e1_));                           \
      PFS_HIP(hipEventRecord(e1_, (st)->s));                   \
      (st)->recs.push_back(KRec{#kern, e0_, e1_});             \
    }                                                          \
  } while (0)

// ---------------------------------------------------------------- runtime
__global__ void publish_k(PubSet p, u32 n, u32* flag, u32 tag) {
  for (u32 q = 0; q < n; q++)
    for (u32 i = threadIdx.x; i < p.words[q]; i += 64) p.dst[q][i] = p.src[q][i];
  if (!flag) return;
  __threadfence_system();
  if (threadIdx.x == 0) __hip_atomic_store(flag, tag, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
static void pub_flush(Stream* st, bool flagged) {
  const u32 n = st->npub;
  st->npub = 0;  // first: the launch below is itself an operation on the stream
  if (flagged) st->tag++;
  publish_k<<<1, 64, 0, st->s>>>(st->pub, n, flagged ? st->flag : nullptr, st->tag);
  LAUNCH_CHECK();
}
// waits for the flag of the gathered reads, giving the core away between
// polls once the wait is longer than a launch; false when it is not there
// after 20 ms (a long queue, or a device error): the caller waits for the
// stream, which reports errors.  (Giving up after 0.3 ms cost a call on 10M
// variables, which waits for millisecond kernels, 0.13 ms.)
static bool pub_wait(Stream* st) {
  pub_flush(st, true);
  const auto t0 = std::chrono::steady_clock::now();
  while (true) {
    for (int i = 0; i < 256; i++)
      if (__atomic_load_n(st->flag, __ATOMIC_ACQUIRE) == st->tag) return true;
    const auto dt = std::chrono::steady_clock::now() - t0;
    if (dt > std::chrono::milliseconds(20)) return false;
    if (dt > std::chrono::microseconds(50)) std::this_thread::yield();
  }
}
static void staging_retain();
static void staging_release();
Stream* stream_create(int device) {
  PFS_HIP(hipSetDevice(device));
  Stream* st = new Stream();
  st->device = device;
  PFS_HIP(hipStreamCreateWithFlags(&st->s, hipStreamNonBlocking));
  if (hipHostMalloc((void**)&st->pin, PIN_BYTES + 256, hipHostMallocCoherent) != hipSuccess) st->pin = nullptr;
  if (st->pin) {
    st->flag = (u32*)(st->pin + PIN_BYTES);
    *st->flag = 0;
  }
  staging_retain();
  return st;
}
void prof_enable(Stream* st, bool on) { st->prof = on; }
void stream_bind(Stream* st) { PFS_HIP(hipSetDevice(st->device)); }
void prof_collect(Stream* st, std::vector<KernelTime>& out) {
  stream_op(st);
  PFS_HIP(hipStreamSynchronize(st->s));
  pin_flush(st);
  std::map<std::string, size_t> idx;
  for (size_t i = 0; i < out.size(); i++) idx[out[i].name] = i;
  for (const KRec& r : st->recs) {
    float ms = 0;
    PFS_HIP(hipEventElapsedTime(&ms, r.a, r.b));
    (void)hipEventDestroy(r.a);
    (void)hipEventDestroy(r.b);
    auto it = idx.find(r.name);
    if (it == idx.end()) {
      idx[r.name] = out.size();
      out.push_back(KernelTime{r.name, 0.0, 0});
      it = idx.find(r.name);
    }
    out[it->second].ms += ms;
    out[it->second].launches++;
  }
  st->recs.clear();
}
void stream_destroy(Stream* st) {
  if (!st) return;
  for (const KRec& r : st->recs) {
    (void)hipEventDestroy(r.a);
    (void)hipEventDestroy(r.b);
  }
  (void)hipStreamSynchronize(st->s);
  // staged reads still pending here belong to a call that ended with an
  // error: their destinations may be gone, so they are dropped
  st->pend.clear();
  if (st->pin) (void)hipHostFree(st->pin);
  (void)hipStreamDestroy(st->s);
  delete st;
  staging_release();
}
void stream_sync(Stream* st) {
  if (st->npub && pub_wait(st)) {  // the flag follows everything queued before it
    pin_flush(st);
    return;
  }
  const hipError_t e = hipStreamSynchronize(st->s);
  if (e != hipSuccess) {
    // the staged reads did not complete: drop them (their destinations are
    // locals of frames the exception unwinds), then report
    st->npub = 0;
    st->pend.clear();
    st->pin_used = 0;
    throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e) + " at " + __FILE__ + ":" +
                             std::to_string(__LINE__));
  }
  pin_flush(st);
}
bool stream_quiesce(Stream* st) {
  if (!st) return true;
  st->npub = 0;
  const bool ok = hipStreamSynchronize(st->s) == hipSuccess;
  if (!ok) (void)hipGetLastError();
  st->pend.clear();
  st->pin_used = 0;
  return ok;
}
void* dev_alloc(size_t bytes) {
  void* p = nullptr;
  if (bytes == 0) bytes = 256;
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    throw std::bad_alloc();
  }
  return p;
}
void dev_free(void* p) {
  if (p) (void)hipFree(p);
}
// small host-to-device copies go through the same pinned area (the host
// data is copied there first; the area is reused only after stream_sync)
void h2d(void* dst, const void* src, size_t bytes, Stream* st) {
  if (!bytes) return;
  stream_op(st);
  if (st->pin && bytes <= PIN_SMALL) {
    if (st->pin_used + bytes > PIN_BYTES) stream_sync(st);
    memcpy(st->pin + st->pin_used, src, bytes);
    PFS_HIP(hipMemcpyAsync(dst, st->pin + st->pin_used, bytes, hipMemcpyHostToDevice, st->s));
    st->pin_used += (bytes + 15) & ~(size_t)15;
    return;
  }
  PFS_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st->s));
}
// Large downloads.  The caller's buffers are pageable as a rule: the runtime
// moves such a copy at 18 GB/s, and the 134 MB of a 4.4M-clause result took 7.8
// ms.  (Into pinned buffers it moves 57 GB/s, and they are left to it: 133 MB
// take 2.5 ms, 3.05 through the ring.)  They go through a ring of pinned slots
// instead: the calling thread keeps the copies into the slots going, and a few
// threads, which live as long as the call, each move their share of every slot
// that has arrived to the caller's memory (one thread moves about 10 GB/s, the
// link 57, so it takes several; page faults of a fresh buffer are shared out
// with them).
// Into buffers used before, 134 MB take 3.3 ms and 290 MB 5.9 instead of 7.8
// and 14.5 (slots of 1 / 2 / 4 MiB: 8.6 / 6.8 / 5.9 ms; 4, 6 and 8 threads
// alike).
// The ring is one per process, made by the first large download, used by one
// call at a time (a second one copies directly, as does one that cannot start
// the threads) and given back with the last stream.
constexpr size_t STG_SLOT = 4 << 20, STG_MIN = 4 << 20;
constexpr u32 STG_SLOTS = 4, STG_THREADS = 4;
struct Staging {
  std::mutex use;  // held by the call that works with the ring
  unsigned char* p = nullptr;
  hipEvent_t ev[STG_SLOTS] = {};
  int device = -1;  // of the events
  void drop() {
    if (!p) return;
    for (hipEvent_t& e : ev)
      if (e) (void)hipEventDestroy(e), e = nullptr;
    (void)hipHostFree(p);
    p = nullptr;
  }
  bool make(int dev) {
    if (p && device == dev) return true;
    drop();
    if (hipHostMalloc((void**)&p, STG_SLOT * STG_SLOTS, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
      return false;
    }
    device = dev;
    for (hipEvent_t& e : ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        drop();
        return false;
      }
    return true;
  }
};
static Staging g_staging;
static std::mutex g_streams_m;
static u32 g_streams = 0;  // streams alive: the last one gives the ring back
static void staging_retain() {
  std::lock_guard<std::mutex> lk(g_streams_m);
  g_streams++;
}
static void staging_release() {
  std::lock_guard<std::mutex> lk(g_streams_m);
  if (--g_streams) return;
  std::lock_guard<std::mutex> use(g_staging.use);
  g_staging.drop();
}
// the ring as staged_copy drives it
struct StagingRing {
  u32 slots;
  hipStream_t s;
  std::atomic<hipError_t> err{hipSuccess};  // the first one
  bool ok(hipError_t e) {
    hipError_t none = hipSuccess;
    if (e != hipSuccess) err.compare_exchange_strong(none, e);
    return e == hipSuccess;
  }
  const unsigned char* slot(u32 k) { return g_staging.p + k * STG_SLOT; }
  bool queue(u32 k, const StagedPiece& c) {
    return ok(hipMemcpyAsync(g_staging.p + k * STG_SLOT, c.src, c.bytes, hipMemcpyDeviceToHost, s)) &&
           ok(hipEventRecord(g_staging.ev[k], s));
  }
  bool arrived(u32 k) { return ok(hipEventSynchronize(g_staging.ev[k])); }
  template <class F>
  std::thread run(F f) {
    return std::thread(f);
  }
};
// ordinary host memory, which a direct copy fills slowly (pinned, managed and
// device memory it fills at the link's rate)
static bool pageable(const void* p) {
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, p) == hipSuccess) return at.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}
void d2h_set(const D2H* set, u32 n, Stream* st) {
  stream_op(st);
  const auto direct = [&](const D2H& c) {
    if (c.bytes) PFS_HIP(hipMemcpyAsync(c.dst, c.src, c.bytes, hipMemcpyDeviceToHost, st->s));
  };
  size_t total = 0, slow = 0;
  for (u32 i = 0; i < n; i++) total += set[i].bytes;
  u32 staged = 0;  // bit i: set[i] goes through the ring
  for (u32 i = 0; i < n && total >= STG_MIN; i++)
    if (set[i].bytes && pageable(set[i].dst)) staged |= 1u << i, slow += set[i].bytes;
  std::unique_lock<std::mutex> lk(g_staging.use, std::defer_lock);
  const u32 nthr = std::min(STG_THREADS, std::max(1u, std::thread::hardware_concurrency() / 2));
  if (slow < STG_MIN || nthr < 2 || !lk.try_lock() || !g_staging.make(st->device)) staged = 0;
  std::vector<StagedPiece> pc;
  for (u32 i = 0; i < n; i++) {
    if (!(staged >> i & 1)) direct(set[i]);
    else
      for (size_t o = 0; o < set[i].bytes; o += STG_SLOT)
        pc.push_back({(char*)set[i].dst + o, (const char*)set[i].src + o, std::min(STG_SLOT, set[i].bytes - o)});
  }
  if (!staged) return;
  StagingRing ring{STG_SLOTS, st->s};
  const Staged r = staged_copy(pc, nthr, ring);
  if (r == Staged::NOT_STARTED)
    for (u32 i = 0; i < n; i++)
      if (staged >> i & 1) direct(set[i]);
  if (r != Staged::FAILED) return;
  (void)hipStreamSynchronize(st->s);  // nothing writes to the slots any more
  throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(ring.err.load()) + " in a staged download");
}
void d2h(void* dst, const void* src, size_t bytes, Stream* st) {
  if (!bytes) return;
  if (bytes >= STG_MIN) {
    const D2H one{dst, src, bytes};
    d2h_set(&one, 1, st);
    return;
  }
  if (st->pin && bytes <= PIN_SMALL) {
    if (st->pin_used + bytes > PIN_BYTES) stream_sync(st);
    if (bytes <= PUB_BYTES && (bytes & 3) == 0 && ((uintptr_t)src & 3) == 0) {
      if (st->npub == PUB_MAX) pub_flush(st, false);
      st->pub.src[st->npub] = (const u32*)src;
      st->pub.dst[st->npub] = (u32*)(st->pin + st->pin_used);
      st->pub.words[st->npub++] = (u32)(bytes / 4);
      st->pend.push_back(PinCopy{dst, st->pin_used, bytes});
      st->pin_used += (bytes + 15) & ~(size_t)15;
      return;
    }
    stream_op(st);
    PFS_HIP(hipMemcpyAsync(st->pin + st->pin_used, src, bytes, hipMemcpyDeviceToHost, st->s));
    st->pend.push_back(PinCopy{dst, st->pin_used, bytes});
    st->pin_used += (bytes + 15) & ~(size_t)15;
    return;
  }
  stream_op(st);
  PFS_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st->s));
}
void d2d(void* dst, const void* src, size_t bytes, Stream* st) {
  stream_op(st);
  if (bytes) PFS_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, st->s));
}
// 16 bytes per thread: one 16-byte store where the address allows it
__global__ void fill_u32_k(u32* d, u32 v, size_t n) {
  const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i + 4 <= n && ((uintptr_t)(d + i) & 15u) == 0) {
    *(uint4*)(d + i) = make_uint4(v, v, v, v);
    return;
  }
  for (size_t k = i; k < n && k < i + 4; k++) d[k] = v;
}
__global__ void fill_u8_k(u8* d, u8 v, size_t n) {
  const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 16;
  if (i + 16 <= n && ((uintptr_t)(d + i) & 15u) == 0) {
    const u32 w = v * 0x01010101u;
    *(uint4*)(d + i) = make_uint4(w, w, w, w);
    return;
  }
  for (size_t k = i; k < n && k < i + 16; k++) d[k] = v;
}
void fill_u32(u32* dst, u32 value, size_t n, Stream* st) {
  if (!n) return;
  KLAUNCH(fill_u32_k, grid_for((n + 3) / 4, 256), 256, st, dst, value, n);
}
void fill_u8(u8* dst, u8 value, size_t n, Stream* st) {
  if (!n) return;
  KLAUNCH(fill_u8_k, grid_for((n + 15) / 16, 256), 256, st, dst, value, n);
}
// several buffers cleared by one launch, 4 KiB of one to a workgroup
struct ZeroSet {
  u8* p[ZERO_PARTS];
  size_t n[ZERO_PARTS];
  u32 end[ZERO_PARTS];  // past a buffer's last workgroup
};
__global__ void __launch_bounds__(256) zero_set_k(ZeroSet z) {
  u32 q = 0;
  while (blockIdx.x >= z.end[q]) q++;  // the last one ends the grid
  u8* d = z.p[q];
  const size_t n = z.n[q], i = ((size_t)(blockIdx.x - (q ? z.end[q - 1] : 0)) * 256 + threadIdx.x) * 16;
  if (i + 16 <= n && ((uintptr_t)(d + i) & 15u) == 0) *(uint4*)(d + i) = make_uint4(0, 0, 0, 0);
  else
    for (size_t k = i; k < n && k < i + 16; k++) d[k] = 0;
}
void zero_set(const ZeroPart (&part)[ZERO_PARTS], Stream* st) {
  ZeroSet z;
  u32 end = 0;
  for (u32 q = 0; q < ZERO_PARTS; q++) {
    z.p[q] = (u8*)part[q].p;
    z.n[q] = part[q].bytes;
    z.end[q] = end += (u32)((part[q].bytes + 4095) / 4096);
  }
  if (end) KLAUNCH(zero_set_k, end, 256, st, z);
}
struct Marker {
  hipEvent_t e;
};
Marker* marker_record(Stream* st) {
  stream_op(st);
  Marker* m = new Marker();
  PFS_HIP(hipEventCreateWithFlags(&m->e, hipEventDisableTiming));
  PFS_HIP(hipEventRecord(m->e, st->s));
  return m;
}
bool marker_done(Marker* m) {
  const hipError_t e = hipEventQuery(m->e);
  if (e == hipErrorNotReady) return false;
  if (e != hipSuccess) (void)hipGetLastError();
  return true;
}
void marker_wait(Marker* m) {
  if (hipEventSynchronize(m->e) != hipSuccess) (void)hipGetLastError();
}
void marker_free(Marker* m) {
  if (!m) return;
  (void)hipEventDestroy(m->e);
  delete m;
}
bool stream_wait(Stream* st) {
  stream_op(st);
  if (hipStreamSynchronize(st->s) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}
void dev_mem_info(size_t* fr, size_t* tot) {
  if (hipMemGetInfo(fr, tot) != hipSuccess) {
    (void)hipGetLastError();
    *fr = *tot = 0;
  }
}
Event* event_record(Stream* st) {
  stream_op(st);
  Event* e = new Event();
  PFS_HIP(hipEventCreate(&e->e));
  PFS_HIP(hipEventRecord(e->e, st->s));
  return e;
}
float event_ms(Event* a, Event* b) {
  PFS_HIP(hipEventSynchronize(b->e));
  float ms = 0;
  PFS_HIP(hipEventElapsedTime(&ms, a->e, b->e));
  return ms;
}
void event_free(Event* e) {
  if (!e) return;
  (void)hipEventDestroy(e->e);
  delete e;
}
const char* device_name(int device) {
  static hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) return "unknown";
  return prop.name;
}
int device_count() {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

// ---------------------------------------------------------------- block scan
constexpr int ST = 256;          // threads per scan workgroup
constexpr int SIPT = 8;          // items per thread
constexpr int STILE = ST * SIPT; // items per workgroup
constexpr int NW = ST / 64;      // wavefronts per workgroup

// exclusive scan of one value per thread over the workgroup; *total gets
// the workgroup sum.  'lw' holds NW words of LDS.
template <int W>  // wavefronts per workgroup
__device__ inline u32 block_excl_scan_w(u32 v, u32* lw, u32* total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  u32 x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const u32 y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) lw[wid] = x;
  __syncthreads();
  u32 pre = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < W; w++) {
    const u32 s = lw[w];
    pre += (w < wid) ? s : 0u;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return pre + x - v;
}
__device__ inline u32 block_excl_scan(u32 v, u32* lw, u32* total) { return block_excl_scan_w<NW>(v, lw, total); }

// order-free compaction: each thread holds the keep bits of SIPT
// consecutive items; the workgroup reserves its slots with one atomic and
// returns each thread's first slot
__device__ inline u32 block_reserve(u32 bits, u32* lw, u32* counter) {
  __shared__ u32 base;
  u32 tot;
  const u32 pre = block_excl_scan(__popc(bits), lw, &tot);
  if (threadIdx.x == 0) base = tot ? atomicAdd(counter, tot) : 0u;
  __syncthreads();
  return base + pre;
}
// grid-stride reductions: a bounded number of workgroups, one atomic per
// wavefront, so a single result word never sees more than a few thousand
// atomics
constexpr unsigned RED_BLOCKS = 1024;
__device__ inline u32 wave_max(u32 x) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) x = max(x, (u32)__shfl_xor(x, d, 64));
  return x;
}
__device__ inline unsigned long long wave_sum64(unsigned long long x) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
  return x;
}
// Long scans: each workgroup covers SCAN_SUB tiles of STILE items (one
// partial sum per workgroup, so the single-workgroup pass over the partials
// stays short); a thread's SIPT consecutive items move as two 16-byte
// loads and stores when the arrays are 16-byte aligned (VEC).
constexpr int SCAN_SUB = 4;
constexpr size_t SBLK = (size_t)STILE * SCAN_SUB;
template <bool VEC>
__device__ inline void load_items(const u32* in, size_t b, size_t n, u32 (&v)[SIPT]) {
  if (VEC && b + SIPT <= n) {
    const uint4 x = *(const uint4*)(in + b), y = *(const uint4*)(in + b + 4);
    v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w, v[4] = y.x, v[5] = y.y, v[6] = y.z, v[7] = y.w;
    return;
  }
#pragma unroll
  for (int i = 0; i < SIPT; i++) v[i] = (b + i < n) ? in[b + i] : 0u;
}
template <bool VEC>
__device__ inline void store_items(u32* out, size_t b, size_t n, const u32 (&v)[SIPT]) {
  if (VEC && b + SIPT <= n) {
    *(uint4*)(out + b) = make_uint4(v[0], v[1], v[2], v[3]);
    *(uint4*)(out + b + 4) = make_uint4(v[4], v[5], v[6], v[7]);
    return;
  }
#pragma unroll
  for (int i = 0; i < SIPT; i++)
    if (b + i < n) out[b + i] = v[i];
}
static_assert(SIPT == 8, "two 16-byte moves per thread");
// up to three arrays of n items scanned by the same launches, one per row
// of the grid
struct ScanSet {
  const u32* in[3];
  u32* out[3];
  u32* total[3];
};
template <bool VEC>
__global__ void scan_reduce_k(ScanSet a, size_t n, u32* part) {
  const u32* in = a.in[blockIdx.y];
  part += (size_t)blockIdx.y * gridDim.x;
  __shared__ u32 lw[NW];
  u32 s = 0;
#pragma unroll
  for (int q = 0; q < SCAN_SUB; q++) {
    u32 v[SIPT];
    load_items<VEC>(in, (size_t)blockIdx.x * SBLK + (size_t)q * STILE + (size_t)threadIdx.x * SIPT, n, v);
#pragma unroll
    for (int i = 0; i < SIPT; i++) s += v[i];
  }
  u32 tot;
  block_excl_scan(s, lw, &tot);
  if (threadIdx.x == 0) part[blockIdx.x] = tot;
}
// exclusive scan of the workgroup partials by one workgroup
__global__ void scan_top_k(u32* part, size_t nb, ScanSet a) {
  u32* total = a.total[blockIdx.x];
  part += (size_t)blockIdx.x * nb;
  __shared__ u32 lw[NW];
  u32 carry = 0;
  for (size_t base = 0; base < nb; base += STILE) {
    const size_t b = base + (size_t)threadIdx.x * SIPT;
    u32 v[SIPT];
    u32 s = 0;
#pragma unroll
    for (int i = 0; i < SIPT; i++) {
      v[i] = (b + i < nb) ? part[b + i] : 0u;
      s += v[i];
    }
    u32 tot;
    u32 pre = block_excl_scan(s, lw, &tot) + carry;
#pragma unroll
    for (int i = 0; i < SIPT; i++) {
      if (b + i < nb) part[b + i] = pre;
      pre += v[i];
    }
    carry += tot;
  }
  if (threadIdx.x == 0 && total) *total = carry;
}
// each thread reads its items before the tile's barriers and writes them
// after, so in == out is fine
template <bool VEC>
__global__ void scan_down_k(ScanSet a, size_t n, const u32* part) {
  const u32* in = a.in[blockIdx.y];
  u32* out = a.out[blockIdx.y];
  part += (size_t)blockIdx.y * gridDim.x;
  __shared__ u32 lw[NW];
  u32 carry = part[blockIdx.x];
#pragma unroll 1
  for (int q = 0; q < SCAN_SUB; q++) {
    const size_t base = (size_t)blockIdx.x * SBLK + (size_t)q * STILE + (size_t)threadIdx.x * SIPT;
    u32 v[SIPT];
    load_items<VEC>(in, base, n, v);
    u32 s = 0;
#pragma unroll
    for (int i = 0; i < SIPT; i++) s += v[i];
    u32 tot;
    u32 pre = block_excl_scan(s, lw, &tot) + carry;
#pragma unroll
    for (int i = 0; i < SIPT; i++) {
      const u32 x = v[i];
      v[i] = pre;
      pre += x;
    }
    store_items<VEC>(out, base, n, v);
    carry += tot;
  }
}
// Short scans in one launch by one workgroup of 1024 threads.  Every thread
// loads all its items (8, 32 or 64 consecutive ones, as 16-byte words where
// both arrays allow it) before the one prefix sum over the workgroup, so the
// launch waits for memory once; walking 32,768 items in four tiles, each
// with its loads, barriers and stores, took 11 us against 5.  Every item is
// read before the barriers and written after, so in == out is fine.
constexpr int S1_T = 1024;
constexpr size_t S1_MAX = 64 * (size_t)S1_T;
template <int IPT, bool VEC>
__global__ void __launch_bounds__(S1_T) scan_one_k(ScanSet a, u32 n) {
  const u32* in = a.in[blockIdx.x];
  u32 *out = a.out[blockIdx.x], *total = a.total[blockIdx.x];
  __shared__ u32 lw[S1_T / 64];
  const u32 b = threadIdx.x * IPT;
  u32 v[IPT / 8][8], s = 0, tot;
#pragma unroll
  for (int q = 0; q < IPT / 8; q++) load_items<VEC>(in, b + 8 * q, n, v[q]);
#pragma unroll
  for (int q = 0; q < IPT / 8; q++)
#pragma unroll
    for (int i = 0; i < 8; i++) s += v[q][i];
  u32 pre = block_excl_scan_w<S1_T / 64>(s, lw, &tot);
#pragma unroll
  for (int q = 0; q < IPT / 8; q++) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const u32 x = v[q][i];
      v[q][i] = pre;
      pre += x;
    }
    store_items<VEC>(out, b + 8 * q, n, v[q]);
  }
  if (threadIdx.x == 0 && total) *total = tot;
}
size_t scan_tmp_bytes(size_t n) { return (grid_for(n, SBLK) + 64) * sizeof(u32); }
template <bool VEC>
static void scan_rows(const ScanSet& a, u32 rows, size_t n, void* tmp, Stream* st) {
  if (n <= S1_MAX) {
    if (n <= 8 * S1_T) KLAUNCH((scan_one_k<8, VEC>), rows, S1_T, st, a, (u32)n);
    else if (n <= 32 * S1_T) KLAUNCH((scan_one_k<32, VEC>), rows, S1_T, st, a, (u32)n);
    else KLAUNCH((scan_one_k<64, VEC>), rows, S1_T, st, a, (u32)n);
    return;
  }
  const unsigned nb = grid_for(n, SBLK);
  u32* part = (u32*)tmp;
  KLAUNCH(scan_reduce_k<VEC>, dim3(nb, rows), ST, st, a, n, part);
  KLAUNCH(scan_top_k, rows, ST, st, part, nb, a);
  KLAUNCH(scan_down_k<VEC>, dim3(nb, rows), ST, st, a, n, part);
}
static void scan_set(const ScanSet& a, u32 rows, size_t n, void* tmp, Stream* st) {
  uintptr_t bits = 0;
  for (u32 q = 0; q < rows; q++) bits |= (uintptr_t)a.in[q] | (uintptr_t)a.out[q];
  if ((bits & 15) == 0) scan_rows<true>(a, rows, n, tmp, st);
  else scan_rows<false>(a, rows, n, tmp, st);
}
void scan_u32(const u32* in, u32* out, size_t n, u32* total, void* tmp, Stream* st) {
  if (n == 0) {
    if (total) fill_u32(total, 0, 1, st);
    return;
  }
  scan_set(ScanSet{{in}, {out}, {total}}, 1, n, tmp, st);
}
// tmp: 3 * scan_tmp_bytes(n)
void scan3_u32(const u32* const (&in)[3], u32* const (&out)[3], size_t n, u32* total, void* tmp, Stream* st) {
  if (n == 0) {
    fill_u32(total, 0, 3, st);
    return;
  }
  scan_set(ScanSet{{in[0], in[1], in[2]}, {out[0], out[1], out[2]}, {total, total + 1, total + 2}}, 3, n, tmp, st);
}

// ---------------------------------------------------------------- stable radix sort
// LSD passes of up to 8 bits.  A pass counts each tile's digits (rs_count_k),
// scans the digit-major counts, then every tile sorts itself by the digit
// in LDS with stable two-bit splits and writes each digit's run to its
// place (rs_scatter_k), so the stores go out in runs rather than one
// scattered word per item.
constexpr int RS_T = 256, RS_IPT = 8, RS_TILE = RS_T * RS_IPT;  // threads, items per thread, items per tile
constexpr int RB = 8, RBUCK = 1 << RB;
static_assert(RS_T == RBUCK, "one digit bin per thread");

// Stable splits by two bits at a time: the four counts of a thread's items
// are 16-bit fields of one 64-bit word, so one prefix sum over the workgroup
// serves both bits.
template <int W>
__device__ inline u64 block_excl_scan64_w(u64 v, u64* lw, u64* total) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  u64 x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const u64 y = __shfl_up((unsigned long long)x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) lw[wid] = x;
  __syncthreads();
  u64 pre = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < W; w++) {
    const u64 s = lw[w];
    pre += (w < wid) ? s : 0ull;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return pre + x - v;
}
// A thread's consecutive items sit IPT words apart from its neighbour's: one
// word of padding per 32 keeps the 64 lanes off a few banks.
__device__ __host__ constexpr u32 lpad(u32 j) { return j + (j >> 5); }
// where this thread's items go in a stable split of the workgroup's items by
// the two bits d[i]
template <int T, int IPT>
__device__ inline void split4(const u32 (&d)[IPT], u32 (&dst)[IPT], u64* lw) {
  static_assert(T * IPT < 65536, "counts are 16-bit fields");
  u64 c = 0, tot;
#pragma unroll
  for (int i = 0; i < IPT; i++) c += 1ull << (16 * d[i]);
  u64 at = block_excl_scan64_w<T / 64>(c, lw, &tot);
  // each field also starts behind the items of the smaller digits
  const u64 t0 = tot & 0xFFFF, t1 = (tot >> 16) & 0xFFFF, t2 = (tot >> 32) & 0xFFFF;
  at += (t0 << 16) + ((t0 + t1) << 32) + ((t0 + t1 + t2) << 48);
#pragma unroll
  for (int i = 0; i < IPT; i++) {
    dst[i] = (u32)(at >> (16 * d[i])) & 0xFFFFu;
    at += 1ull << (16 * d[i]);
  }
}
__global__ void __launch_bounds__(RS_T) rs_count_k(const u32* keys, size_t n, int shift, u32 mask, u32* counts,
                                                  u32 nb) {
  __shared__ u32 h[RBUCK];
  h[threadIdx.x] = 0;  // RS_T == RBUCK
  __syncthreads();
  const size_t base = (size_t)blockIdx.x * RS_TILE;
#pragma unroll
  for (int i = 0; i < RS_IPT; i++) {
    const size_t j = base + (size_t)i * RS_T + threadIdx.x;
    if (j < n) atomicAdd(&h[(keys[j] >> shift) & mask], 1u);
  }
  __syncthreads();
  counts[(size_t)threadIdx.x * nb + blockIdx.x] = h[threadIdx.x];
}
// vin null: the values are the positions; kout null: the sorted keys are
// not wanted; starts: where the digits of q << sshift and more begin, for
// q below nstarts
__global__ void __launch_bounds__(RS_T) rs_scatter_k(const u32* kin, const u32* vin, u32* kout, u32* vout,
                                                    size_t n, int shift, int width, const u32* offs, u32 nb,
                                                    u32* starts, u32 nstarts, int sshift) {
  __shared__ u32 sk[lpad(RS_TILE)], sv[lpad(RS_TILE)];
  __shared__ u32 start[RBUCK];
  __shared__ u32 lw[RS_T / 64];
  __shared__ u64 lw64[RS_T / 64];
  const u32 mask = (1u << width) - 1u;
  const size_t base = (size_t)blockIdx.x * RS_TILE;
  const u32 cnt = (u32)min((size_t)RS_TILE, n - base), j0 = threadIdx.x * RS_IPT;
  // the tile in input order; slots past the input take the largest digit
  // and stay behind every item (they come last and the splits are stable)
#pragma unroll
  for (int i = 0; i < RS_IPT; i++) {
    const u32 j = i * RS_T + threadIdx.x;
    sk[lpad(j)] = j < cnt ? kin[base + j] : (mask << shift);
    sv[lpad(j)] = j < cnt ? (vin ? vin[base + j] : (u32)(base + j)) : 0u;
  }
  if (blockIdx.x == 0 && threadIdx.x < nstarts) {
    const u32 q = threadIdx.x << sshift;
    starts[threadIdx.x] = q <= mask ? offs[(size_t)q * nb] : (u32)n;
  }
  start[threadIdx.x] = 0;
  __syncthreads();
  // thread t moves items t*IPT .. t*IPT+IPT-1
  for (int bit = 0; bit < width; bit += 2) {
    u32 k[RS_IPT], v[RS_IPT], d[RS_IPT], dst[RS_IPT];
#pragma unroll
    for (int i = 0; i < RS_IPT; i++) {
      k[i] = sk[lpad(j0 + i)];
      v[i] = sv[lpad(j0 + i)];
      d[i] = (k[i] >> (shift + bit)) & (bit + 1 < width ? 3u : 1u);
    }
    split4<RS_T, RS_IPT>(d, dst, lw64);  // its barriers follow every read above
#pragma unroll
    for (int i = 0; i < RS_IPT; i++) {
      sk[lpad(dst[i])] = k[i];
      sv[lpad(dst[i])] = v[i];
    }
    __syncthreads();
  }
  // where each digit's run starts in the sorted tile
#pragma unroll
  for (int i = 0; i < RS_IPT; i++) {
    const u32 j = i * RS_T + threadIdx.x;
    if (j < cnt) atomicAdd(&start[(sk[lpad(j)] >> shift) & mask], 1u);
  }
  __syncthreads();
  u32 tot;
  const u32 c = start[threadIdx.x];
  const u32 pre = block_excl_scan_w<RS_T / 64>(c, lw, &tot);
  start[threadIdx.x] = pre;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RS_IPT; i++) {
    const u32 j = i * RS_T + threadIdx.x;
    if (j < cnt) {
      const u32 key = sk[lpad(j)], d = (key >> shift) & mask;
      const u32 dst = offs[(size_t)d * nb + blockIdx.x] + (j - start[d]);
      if (kout) kout[dst] = key;
      vout[dst] = sv[lpad(j)];
    }
  }
}
size_t radix_tmp_bytes(size_t n) {
  const size_t nb = grid_for(n ? n : 1, RS_TILE);
  return 2 * n * sizeof(u32) + RBUCK * nb * sizeof(u32) + scan_tmp_bytes(RBUCK * nb) + 256;
}
// Sorts of up to SO_MAX items in one launch by one workgroup: T threads
// hold IPT consecutive items each in registers, and stable splits move them
// through LDS.  The three launches and two copies of a pass over digits cost
// 40-60 us whatever the size; this sorts 8,192 items by 8 bits in about 12 us.
// (32 items per thread in one workgroup took 85 us for 20,000 candidates and
// 11-bit keys, two digit passes 54.)
constexpr int SO_T = 1024, SO_IPT = 8;
constexpr u32 SO_MAX = SO_T * SO_IPT;
// values sorted in place by the low 'bits' bits of their keys (the keys stay)
template <int T>
__global__ void __launch_bounds__(T) sort_one_k(const u32* keys, u32* vals, u32 n, int bits) {
  constexpr int IPT = SO_IPT;
  __shared__ u32 sk[lpad(T * IPT)];
  __shared__ uint16_t si[lpad(T * IPT)];
  __shared__ u64 lw[T / 64];
  const u32 j0 = threadIdx.x * IPT;
  u32 k[IPT], id[IPT], d[IPT], dst[IPT], v[IPT];
#pragma unroll
  for (int i = 0; i < IPT; i++) {
    k[i] = j0 + i < n ? keys[j0 + i] : 0xFFFFFFFFu;  // slots past the input stay behind it
    id[i] = j0 + i;
  }
  for (int bit = 0; bit < bits; bit += 2) {
    const u32 m = bit + 1 < bits ? 3u : 1u;
#pragma unroll
    for (int i = 0; i < IPT; i++) d[i] = (k[i] >> bit) & m;
    split4<T, IPT>(d, dst, lw);
#pragma unroll
    for (int i = 0; i < IPT; i++) {
      sk[lpad(dst[i])] = k[i];
      si[lpad(dst[i])] = (uint16_t)id[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IPT; i++) {
      k[i] = sk[lpad(j0 + i)];
      id[i] = si[lpad(j0 + i)];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < IPT; i++) v[i] = j0 + i < n ? vals[id[i]] : 0u;
  __syncthreads();  // every value is read before any is written
#pragma unroll
  for (int i = 0; i < IPT; i++)
    if (j0 + i < n) vals[j0 + i] = v[i];
}
// sorts the values by the low 'bits' bits of their keys (higher bits are
// ignored); the keys are consumed
void radix_sort_pairs(u32* keys, u32* vals, size_t n, int bits, void* tmp, Stream* st) {
  if (n < 2 || bits <= 0) return;
  bits = std::min(bits, 32);
  if (n <= SO_MAX) {
    if (n <= 256 * SO_IPT) KLAUNCH(sort_one_k<256>, 1, 256, st, keys, vals, (u32)n, bits);
    else KLAUNCH(sort_one_k<SO_T>, 1, SO_T, st, keys, vals, (u32)n, bits);
    return;
  }
  const u32 nb = grid_for(n, RS_TILE);
  u32* k2 = (u32*)tmp;
  u32* v2 = k2 + n;
  u32* counts = v2 + n;
  void* stmp = counts + (size_t)RBUCK * nb;
  u32 *ka = keys, *va = vals, *kb = k2, *vb = v2;
  int passes = 0;
  for (int shift = 0; shift < bits; shift += RB) {
    const int width = std::min(RB, bits - shift);
    const u32 mask = (1u << width) - 1u;
    const bool last = shift + RB >= bits;
    KLAUNCH(rs_count_k, nb, RS_T, st, ka, n, shift, mask, counts, nb);
    scan_u32(counts, counts, (size_t)(mask + 1) * nb, nullptr, stmp, st);
    KLAUNCH(rs_scatter_k, nb, RS_T, st, ka, va, last ? nullptr : kb, vb, n, shift, width, counts, nb, nullptr, 0u, 0);
    u32* t = ka; ka = kb; kb = t;
    t = va; va = vb; vb = t;
    passes++;
  }
  if (passes & 1) d2d(vals, va, n * sizeof(u32), st);
}

// ---------------------------------------------------------------- placement by a small key
// The items 0..n-1 in the stable order of a small key (below 1 << bits, at
// most 8 bits) that f computes: out receives f.val(t) in that order,
// starts[q] for q below nstarts where the keys of q << sshift and more
// begin.  zero: nz words cleared on
// the way (counters of the launches that follow).  One launch by one
// workgroup for up to SO_MAX items, else three (keys and their counts per
// tile, one scan, the scatter); what this replaces was a launch for the keys,
// three for the digit pass, two copies, one for the starts and a fill.  (One
// workgroup with 16 or 32 items per thread takes 37 and 116 us for 12,000 and
// 30,000 variables, whose list sizes it reads, the three launches 28 and 30.)
constexpr int KEY_IDX_BITS = 13;
static_assert(SO_MAX <= (1u << KEY_IDX_BITS), "an item's index and key share a word");
template <int T, class F>
__global__ void __launch_bounds__(T) place_one_k(F f, u32 n, int bits, u32* out, u32* starts, u32 nstarts, int sshift,
                                                 u32* zero, u32 nz) {
  constexpr int IPT = SO_IPT;
  __shared__ u32 sk[lpad(T * IPT)];
  __shared__ u64 lw[T / 64];
  if (threadIdx.x < nz) zero[threadIdx.x] = 0;
  const u32 j0 = threadIdx.x * IPT;
  const u32 top = (1u << bits) - 1u, imask = (1u << KEY_IDX_BITS) - 1u;
  u32 x[IPT], d[IPT], dst[IPT];
  // strided for the reads of f; slots past the input take the largest key
  // and stay behind every item (they come last and the splits are stable)
#pragma unroll
  for (int i = 0; i < IPT; i++) {
    const u32 j = i * T + threadIdx.x;
    sk[lpad(j)] = ((j < n ? f.key(j) : top) << KEY_IDX_BITS) | j;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < IPT; i++) x[i] = sk[lpad(j0 + i)];
  __syncthreads();
  for (int bit = 0; bit < bits; bit += 2) {
#pragma unroll
    for (int i = 0; i < IPT; i++) d[i] = (x[i] >> (KEY_IDX_BITS + bit)) & (bit + 1 < bits ? 3u : 1u);
    split4<T, IPT>(d, dst, lw);
#pragma unroll
    for (int i = 0; i < IPT; i++) sk[lpad(dst[i])] = x[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IPT; i++) x[i] = sk[lpad(j0 + i)];
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < IPT; i++) sk[lpad(j0 + i)] = x[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < IPT; i++) {
    const u32 j = i * T + threadIdx.x;
    if (j >= n) continue;
    out[j] = f.val(sk[lpad(j)] & imask);
    if (nstarts) {
      const int sh = KEY_IDX_BITS + sshift;
      const u32 key = sk[lpad(j)] >> sh;
      for (u32 q = j ? (sk[lpad(j - 1)] >> sh) + 1 : 0; q <= key && q < nstarts; q++) starts[q] = j;
      if (j == n - 1)
        for (u32 q = key + 1; q < nstarts; q++) starts[q] = n;
    }
  }
}
template <class F>
__global__ void __launch_bounds__(RS_T) place_count_k(F f, u32 n, u32* keys, u32* vals, u32* counts, u32 ndig, u32 nb,
                                                      u32* zero, u32 nz) {
  __shared__ u32 h[RBUCK];
  if (blockIdx.x == 0 && threadIdx.x < nz) zero[threadIdx.x] = 0;
  h[threadIdx.x] = 0;  // RS_T == RBUCK
  __syncthreads();
  const u32 base = blockIdx.x * RS_TILE;
#pragma unroll
  for (int i = 0; i < RS_IPT; i++) {
    const u32 j = base + i * RS_T + threadIdx.x;
    if (j < n) {
      const u32 k = f.key(j);
      keys[j] = k;
      vals[j] = f.val(j);
      atomicAdd(&h[k], 1u);
    }
  }
  __syncthreads();
  if (threadIdx.x < ndig) counts[(size_t)threadIdx.x * nb + blockIdx.x] = h[threadIdx.x];
}
// tmp: radix_tmp_bytes(n)
template <class F>
void place(F f, u32 n, int bits, u32* out, u32* starts, u32 nstarts, int sshift, u32* zero, u32 nz, void* tmp,
           Stream* st) {
  if (n <= 256 * SO_IPT) {
    KLAUNCH((place_one_k<256, F>), 1, 256, st, f, n, bits, out, starts, nstarts, sshift, zero, nz);
  } else if (n <= SO_MAX) {
    KLAUNCH((place_one_k<SO_T, F>), 1, SO_T, st, f, n, bits, out, starts, nstarts, sshift, zero, nz);
  } else {
    const u32 nb = grid_for(n, RS_TILE), ndig = 1u << bits;
    u32* k2 = (u32*)tmp;
    u32* v2 = k2 + n;
    u32* counts = v2 + n;
    KLAUNCH(place_count_k<F>, nb, RS_T, st, f, n, k2, v2, counts, ndig, nb, zero, nz);
    scan_u32(counts, counts, (size_t)ndig * nb, nullptr, counts + (size_t)RBUCK * nb, st);
    KLAUNCH(rs_scatter_k, nb, RS_T, st, k2, v2, nullptr, out, (size_t)n, 0, bits, counts, nb, starts, nstarts,
            sshift);
  }
}

// Stable sort of the clause order by the list key (size, first literal, last
// literal, signature): the reference's aggresivesort of the result
// (src/cpu/simplify.cpp:263 with CNF_CMP_KEY, simplify.h:29-42; the GPU
// build's stable sort with OLIST_CMP, src/gpu/cnf.cu:232-233).  Four stable
// radix passes over the handles, least significant key first.
__global__ void clause_key_k(const u32* pool, const u32* handles, u32 n, int which, u32* keys) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const u32 c = handles[i];
  const u32 size = hdr_size(pool[c]);
  u32 k;
  if (which == 0) k = pool[c + 1];                                // signature
  else if (which == 1) k = size ? pool[c + CL_HDR + size - 1] : 0;  // last literal
  else if (which == 2) k = size ? pool[c + CL_HDR] : 0;             // first literal
  else k = size;
  keys[i] = k;
}
void k_aggr_sort(const DB& db, u32* keys, void* tmp, Stream* st) {
  const u32 n = db.ncls;
  if (n < 2) return;
  for (int which = 0; which < 4; which++) {
    KLAUNCH(clause_key_k, grid_for(n, 256), 256, st, db.lits, db.c_off, n, which, keys);
    radix_sort_pairs(keys, db.c_off, n, which == 3 ? 24 : 32, tmp, st);
  }
}

// ---------------------------------------------------------------- OT
// clause-parallel kernels run over clause indices and work on the handles
// c_off[i]
__global__ void hist_k(DB db, u32* hist) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls) hist_clause(db, db.c_off[i], hist);
}
__global__ void scatter_k(DB db, u32* cursor) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls) scatter_clause(db, db.c_off[i], cursor);
}
void k_hist(const DB& db, u32* hist, Stream* st) {
  if (!db.ncls) return;
  KLAUNCH(hist_k, grid_for(db.ncls, 256), 256, st, db, hist);
}
void k_scatter(const DB& db, u32* cursor, Stream* st) {
  if (!db.ncls) return;
  KLAUNCH(scatter_k, grid_for(db.ncls, 256), 256, st, db, cursor);
}

// ---------------------------------------------------------------- OT by literal ranges
// The same table without a global atomic per occurrence: the (literal,
// handle) pairs of the live clauses are partitioned by literal range
// (1 << bits literals each, counted per range and tile of clauses, the
// counts scanned range-major), then one workgroup per range counts its
// literals in LDS, scans them into the list offsets (the range's first
// offset is where its partition starts, because the ranges are in literal
// order) and places the handles with LDS cursors.  Order inside a list is
// free, as with the per-occurrence atomics.
constexpr int OTP_UNROLL = 4;
constexpr int OTP_TB = 1024;  // threads per tile workgroup
constexpr u32 OTP_NONE = 0xFFFFFFFFu;  // no clause / no literal in this slot
// calls f(literal, handle) for every literal of the live clauses of the
// tile [c0, c1); each thread holds OTP_UNROLL clauses at a time
template <class F>
__device__ inline void otp_tile(const DB& db, u32 c0, u32 c1, F f) {
  for (u32 i = c0 + threadIdx.x; i < c1; i += OTP_UNROLL * OTP_TB) {
    u32 c[OTP_UNROLL], h[OTP_UNROLL];
#pragma unroll
    for (int q = 0; q < OTP_UNROLL; q++) {
      const u32 ii = i + q * OTP_TB;
      c[q] = ii < c1 ? db.c_off[ii] : OTP_NONE;
    }
#pragma unroll
    for (int q = 0; q < OTP_UNROLL; q++) h[q] = c[q] != OTP_NONE ? db.lits[c[q]] : 0u;
#pragma unroll
    for (int q = 0; q < OTP_UNROLL; q++) {
      if (c[q] == OTP_NONE || st_deleted(hdr_flags(h[q]))) continue;
      const u32* l = db.lits + c[q] + CL_HDR;
      const u32 n = hdr_size(h[q]);
      for (u32 k = 0; k < n; k++) f(l[k], c[q]);
    }
  }
}
// the tile of workgroup b: b itself, or with xcd the tiles taken in runs,
// one run per XCD (workgroups go to the 8 XCDs round robin, so XCD x runs
// the workgroups b = x mod 8; it gets tiles start(x) .. start(x + 1) - 1)
__device__ inline u32 otp_tile_of(u32 b, u32 nblk, int xcd) {
  if (!xcd) return b;
  const u32 q = nblk >> 3, r = nblk & 7u, x = b & 7u;
  return x * q + min(x, r) + (b >> 3);
}
__global__ void __launch_bounds__(OTP_TB) otp_count_k(DB db, u32 ct, int bits, u32 nr, u32 nblk, int xcd,
                                                      u32* counts) {
  extern __shared__ u32 lc[];
  for (u32 j = threadIdx.x; j < nr; j += OTP_TB) lc[j] = 0;
  __syncthreads();
  const u32 t = otp_tile_of(blockIdx.x, nblk, xcd);
  const u32 c0 = t * ct, c1 = min(db.ncls, c0 + ct);
  otp_tile(db, c0, c1, [&](u32 l, u32) { atomicAdd(&lc[l >> bits], 1u); });
  __syncthreads();
  for (u32 j = threadIdx.x; j < nr; j += OTP_TB) counts[(size_t)j * nblk + t] = lc[j];
}
// TABLE: pairs (literal, handle) in one 8-byte word each (one store per
// occurrence); otherwise the literals alone
template <bool TABLE>
__global__ void __launch_bounds__(OTP_TB) otp_part_k(DB db, u32 ct, int bits, u32 nr, u32 nblk, int xcd,
                                                     const u32* offs, void* out) {
  extern __shared__ u32 lc[];
  const u32 t = otp_tile_of(blockIdx.x, nblk, xcd);
  for (u32 j = threadIdx.x; j < nr; j += OTP_TB) lc[j] = offs[(size_t)j * nblk + t];
  __syncthreads();
  const u32 c0 = t * ct, c1 = min(db.ncls, c0 + ct);
  otp_tile(db, c0, c1, [&](u32 l, u32 c) {
    const u32 p = atomicAdd(&lc[l >> bits], 1u);
    if (TABLE)
      ((uint2*)out)[p] = make_uint2(l, c);
    else
      ((u32*)out)[p] = l;
  });
}
// one workgroup per literal range r: literals [r << bits, (r + 1) << bits)
// whose pairs sit at [offs[r * nblk], offs[(r + 1) * nblk]) (the scan's
// total past the last range).  Without TABLE only the counts (hist) are
// written.
constexpr int OTP_LD = 8;
// threads per range workgroup: 1024 (two workgroups per CU) against 256
// (five, bound by the 32 KiB of counters) took the heavy-tailed round's
// range kernel from 2.04 to 1.50 ms and Tseitin's from 0.35 to 0.28 ms:
// more loads in flight per range and fewer table slices open at once per
// XCD; reserving 64 KiB of LDS on top changed nothing
constexpr int OTP_RTB = 1024;
// the lists of a range with at most this many entries are put together in LDS
// and written in one run
constexpr u32 OTP_LISTS = OTP_LD * OTP_RTB;
template <bool TABLE>
__device__ inline void otp_range(const DB& db, int bits, u32 n2, u32 b0, u32 b1, const u32* total, const void* in,
                                 u32* hist, u32* lc, u32* st) {
  const u32* plit = (const u32*)in;
  const uint2* pair = (const uint2*)in;
  __shared__ u32 lw[OTP_RTB / 64];
  const u32 r = blockIdx.x, nl = 1u << bits, base = r << bits;
  for (u32 j = threadIdx.x; j < nl; j += OTP_RTB) lc[j] = 0;
  __syncthreads();
  if (TABLE && b1 - b0 <= OTP_LISTS) {
    const u32 n = b1 - b0, per = nl / OTP_RTB, j0 = threadIdx.x * per;
    uint2 e[OTP_LD];
    u32 at[OTP_LD];
#pragma unroll
    for (int q = 0; q < OTP_LD; q++)
      if (q * OTP_RTB + threadIdx.x < n) e[q] = pair[b0 + q * OTP_RTB + threadIdx.x];
#pragma unroll
    for (int q = 0; q < OTP_LD; q++)
      if (q * OTP_RTB + threadIdx.x < n) at[q] = atomicAdd(&lc[e[q].x - base], 1u);
    __syncthreads();
    u32 s = 0, tot;
    for (u32 k = 0; k < per; k++) s += lc[j0 + k];
    u32 pre = block_excl_scan_w<OTP_RTB / 64>(s, lw, &tot);
    for (u32 k = 0; k < per; k++) {
      const u32 v = lc[j0 + k];
      lc[j0 + k] = pre;
      pre += v;
    }
    __syncthreads();
    for (u32 j = threadIdx.x; j < nl && base + j < n2; j += OTP_RTB) {
      const u32 o = lc[j], sz = (j + 1 < nl ? lc[j + 1] : n) - o;
      db.ot_off[base + j] = b0 + o;
      db.ot_size[base + j] = sz;
      hist[base + j] = sz;
    }
    if (r + 1 == gridDim.x && threadIdx.x == 0) db.ot_off[n2] = *total;
#pragma unroll
    for (int q = 0; q < OTP_LD; q++)
      if (q * OTP_RTB + threadIdx.x < n) st[lc[e[q].x - base] + at[q]] = e[q].y;
    __syncthreads();
    for (u32 j = threadIdx.x; j < n; j += OTP_RTB) db.ot_refs[b0 + j] = st[j];
    return;
  }
  for (u32 p = b0 + threadIdx.x; p < b1; p += OTP_LD * OTP_RTB) {
    u32 l[OTP_LD];
#pragma unroll
    for (int q = 0; q < OTP_LD; q++)
      l[q] = p + q * OTP_RTB < b1 ? (TABLE ? pair[p + q * OTP_RTB].x : plit[p + q * OTP_RTB]) : OTP_NONE;
#pragma unroll
    for (int q = 0; q < OTP_LD; q++)
      if (l[q] != OTP_NONE) atomicAdd(&lc[l[q] - base], 1u);
  }
  __syncthreads();
  if (!TABLE) {
    for (u32 j = threadIdx.x; j < nl; j += OTP_RTB)
      if (base + j < n2) hist[base + j] = lc[j];
    return;
  }
  // exclusive scan: each thread owns nl / OTP_RTB consecutive counters
  const u32 per = nl / OTP_RTB, j0 = threadIdx.x * per;
  u32 s = 0;
  for (u32 k = 0; k < per; k++) s += lc[j0 + k];
  u32 tot;
  u32 pre = block_excl_scan_w<OTP_RTB / 64>(s, lw, &tot) + b0;
  for (u32 k = 0; k < per; k++) {
    const u32 v = lc[j0 + k];
    lc[j0 + k] = pre;
    pre += v;
  }
  __syncthreads();
  for (u32 j = threadIdx.x; j < nl; j += OTP_RTB)
    if (base + j < n2) db.ot_off[base + j] = lc[j];
  if (r + 1 == gridDim.x && threadIdx.x == 0) db.ot_off[n2] = *total;
  // every offset is read out of LDS before any cursor moves
  __syncthreads();
  for (u32 p = b0 + threadIdx.x; p < b1; p += OTP_LD * OTP_RTB) {
    u32 l[OTP_LD], c[OTP_LD];
#pragma unroll
    for (int q = 0; q < OTP_LD; q++) {
      const uint2 e = p + q * OTP_RTB < b1 ? pair[p + q * OTP_RTB] : make_uint2(OTP_NONE, 0u);
      l[q] = e.x;
      c[q] = e.y;
    }
#pragma unroll
    for (int q = 0; q < OTP_LD; q++)
      if (l[q] != OTP_NONE) db.ot_refs[atomicAdd(&lc[l[q] - base], 1u)] = c[q];
  }
  __syncthreads();
  // the cursors end at the next list's offset: size = cursor - offset
  for (u32 j = threadIdx.x; j < nl; j += OTP_RTB)
    if (base + j < n2) {
      const u32 sz = lc[j] - db.ot_off[base + j];
      db.ot_size[base + j] = sz;
      hist[base + j] = sz;
    }
}
template <bool TABLE>
__global__ void __launch_bounds__(OTP_RTB) otp_range_k(DB db, int bits, u32 n2, u32 nblk, const u32* offs,
                                                  const u32* total, const void* in, u32* hist) {
  extern __shared__ u32 lc[];
  __shared__ u32 st[TABLE ? OTP_LISTS : 1];
  const u32 r = blockIdx.x, b0 = offs[(size_t)r * nblk];
  const u32 b1 = r + 1 < gridDim.x ? offs[(size_t)(r + 1) * nblk] : *total;
  otp_range<TABLE>(db, bits, n2, b0, b1, total, in, hist, lc, st);
}

// In two steps for many literals.  One step needs a range per 4,096 or 8,192
// literals: a tile's pairs go to thousands of open lines, which the L2s write
// back a few words at a time, and a range's lists are as scattered.  Here the
// first step fills one line per OTP2_BITS + OTP2_SUB bits of literals, the
// pairs of each such range are partitioned again among its 1 << OTP2_SUB
// parts, and a part's lists are put together in LDS.  10M variables in 40M
// clauses: counts, partition and ranges 0.44 + 1.63 + 1.53 ms in one step;
// 0.30 + 0.88, 0.19 + 0.42 and 0.48 ms here (0.72 and 0.83 for the last two
// without LDS).
//
// tb: the first tile of each range (tiles of OTP2_TILE pairs, none crossing
// ranges), tb[nr] their number
__global__ void __launch_bounds__(OTP2_MAX_RANGES) otp2_tiles_k(const u32* offs, u32 nblk, u32 nr, const u32* total,
                                                               u32* tb) {
  __shared__ u32 lw[OTP2_MAX_RANGES / 64];
  const u32 r = threadIdx.x;
  u32 n = 0, tot;
  if (r < nr) n = (r + 1 < nr ? offs[(size_t)(r + 1) * nblk] : *total) - offs[(size_t)r * nblk];
  const u32 pre = block_excl_scan_w<OTP2_MAX_RANGES / 64>((n + OTP2_TILE - 1) / OTP2_TILE, lw, &tot);
  if (r < nr) tb[r] = pre;
  if (r == 0) tb[nr] = tot;
}
struct Otp2Tile {
  u32 b0, b1;     // its pairs
  u32 at, step;   // its count of part s is word at + s * step
};
__device__ inline bool otp2_tile(u32 t, const u32* offs, u32 nblk, u32 nr, const u32* total, const u32* tb,
                                 Otp2Tile* x) {
  if (t >= tb[nr]) return false;
  u32 lo = 0, hi = nr;  // tb[lo] <= t < tb[hi]
  while (hi - lo > 1) {
    const u32 m = (lo + hi) >> 1;
    if (tb[m] <= t) lo = m;
    else hi = m;
  }
  const u32 end = lo + 1 < nr ? offs[(size_t)(lo + 1) * nblk] : *total;
  x->b0 = offs[(size_t)lo * nblk] + (t - tb[lo]) * OTP2_TILE;
  x->b1 = min(end, x->b0 + OTP2_TILE);
  x->step = tb[lo + 1] - tb[lo];
  x->at = (tb[lo] << OTP2_SUB) + (t - tb[lo]);
  return true;
}
constexpr u32 OTP2_PARTS = 1u << OTP2_SUB;
__global__ void __launch_bounds__(OTP_TB) otp2_count_k(const u32* offs, u32 nblk, u32 nr, const u32* total,
                                                       const u32* tb, const uint2* in, u32* counts) {
  __shared__ u32 lc[OTP2_PARTS];
  Otp2Tile x;
  if (!otp2_tile(blockIdx.x, offs, nblk, nr, total, tb, &x)) return;  // the whole workgroup
  if (threadIdx.x < OTP2_PARTS) lc[threadIdx.x] = 0;
  __syncthreads();
  for (u32 p = x.b0 + threadIdx.x; p < x.b1; p += OTP_LD * OTP_TB) {
    u32 l[OTP_LD];
#pragma unroll
    for (int q = 0; q < OTP_LD; q++) l[q] = p + q * OTP_TB < x.b1 ? in[p + q * OTP_TB].x : OTP_NONE;
#pragma unroll
    for (int q = 0; q < OTP_LD; q++)
      if (l[q] != OTP_NONE) atomicAdd(&lc[(l[q] >> OTP2_BITS) & (OTP2_PARTS - 1)], 1u);
  }
  __syncthreads();
  if (threadIdx.x < OTP2_PARTS) counts[x.at + threadIdx.x * x.step] = lc[threadIdx.x];
}
// the tile in its parts' order in LDS first, so that the stores go out in runs
__global__ void __launch_bounds__(OTP_TB) otp2_part_k(const u32* offs, u32 nblk, u32 nr, const u32* total,
                                                      const u32* tb, const uint2* in, const u32* counts, uint2* out) {
  __shared__ uint2 st[OTP2_TILE];
  __shared__ u32 cnt[OTP2_PARTS], to[OTP2_PARTS];  // to: where a part's run goes, less its place in the tile
  __shared__ u32 lw[OTP_TB / 64];
  Otp2Tile x;
  if (!otp2_tile(blockIdx.x, offs, nblk, nr, total, tb, &x)) return;
  if (threadIdx.x < OTP2_PARTS) cnt[threadIdx.x] = 0;
  __syncthreads();
  constexpr int PT = OTP2_TILE / OTP_TB;
  const u32 n = x.b1 - x.b0;
  uint2 e[PT];
  u32 at[PT];
#pragma unroll
  for (int q = 0; q < PT; q++) {
    const u32 j = q * OTP_TB + threadIdx.x;
    if (j < n) e[q] = in[x.b0 + j];
  }
#pragma unroll
  for (int q = 0; q < PT; q++)
    if (q * OTP_TB + threadIdx.x < n) at[q] = atomicAdd(&cnt[(e[q].x >> OTP2_BITS) & (OTP2_PARTS - 1)], 1u);
  __syncthreads();
  u32 tot;
  const u32 c = threadIdx.x < OTP2_PARTS ? cnt[threadIdx.x] : 0u;
  const u32 pre = block_excl_scan_w<OTP_TB / 64>(c, lw, &tot);
  if (threadIdx.x < OTP2_PARTS) {
    cnt[threadIdx.x] = pre;
    to[threadIdx.x] = counts[x.at + threadIdx.x * x.step] - pre;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PT; q++)
    if (q * OTP_TB + threadIdx.x < n) st[cnt[(e[q].x >> OTP2_BITS) & (OTP2_PARTS - 1)] + at[q]] = e[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PT; q++) {
    const u32 j = q * OTP_TB + threadIdx.x;
    if (j < n) {
      const uint2 v = st[j];
      out[to[(v.x >> OTP2_BITS) & (OTP2_PARTS - 1)] + j] = v;
    }
  }
}
// a workgroup per part
__global__ void __launch_bounds__(OTP_RTB) otp2_range_k(DB db, u32 n2, const u32* tb, const u32* counts,
                                                        const u32* total, const uint2* in, u32* hist) {
  __shared__ u32 lc[1 << OTP2_BITS], st[OTP_LISTS];
  const u32 r = blockIdx.x >> OTP2_SUB, s = blockIdx.x & (OTP2_PARTS - 1), step = tb[r + 1] - tb[r];
  const u32 at = (tb[r] << OTP2_SUB) + s * step;  // the next part starts where the next word says
  otp_range<true>(db, OTP2_BITS, n2, counts[at], counts[at + step], total, in, hist, lc, st);
}
bool otp_plan(size_t n2, size_t ncls, OtpPlan* p, int tile_log2, int xcd) {
  // LDS per workgroup: nr words in the tile kernels (up to 48 KiB); in the
  // range kernel 1 << bits words, and for a table the 32 KiB in which a range's
  // lists are put together: 64 KiB and 64 bytes for ranges of 8,192 literals,
  // of the 160 KiB that a workgroup may have on gfx950.  Ranges of 1,024 literals while
  // there are few enough of them: a workgroup each, and a range's lists fit
  // its LDS (against 4,096 in all cases, the range kernel took 9 instead of
  // 29 us for 77,777 variables, 20 instead of 56 for 300,000, 25 instead of
  // 67 for 500,000, the tile kernels as long as before); of 8192 literals
  // once ranges of 4096 would number 2048 or more
  int bits = 10;
  while (bits < 12 && (n2 >> bits) >= 1024) bits++;
  if ((n2 >> bits) >= 2048) bits = 13;
  const size_t nr = (n2 + ((size_t)1 << bits) - 1) >> bits;
  if (nr > OTP_MAX_RANGES || ncls == 0) return false;
  // tiles of 32 clauses per 4,096 literals (longer segments of pairs for
  // the partition's writes, fewer counts), at most 16,384 clauses: on the
  // heavy-tailed round (2,442 ranges) tiles of 16,384 clauses instead of
  // 131,072 gave 2,442 workgroups instead of 306 and took the count and
  // partition kernels from 0.56 + 2.69 to 0.38 + 2.24 ms
  size_t ct = 4096;
  while (ct < 32 * (n2 >> 12) && ct < 16384) ct <<= 1;
  if (tile_log2 >= 10) ct = (size_t)1 << tile_log2;
  p->xcd = xcd;
  p->bits = bits;
  p->nr = (u32)nr;
  p->ct = (u32)ct;
  p->nblk = (u32)((ncls + ct - 1) / ct);
  p->ncounts = (size_t)p->nr * p->nblk;
  return true;
}
bool otp_plan2(size_t n2, size_t ncls, size_t pairs, OtpPlan* p, int tile_log2, int xcd) {
  constexpr int bits = OTP2_BITS + OTP2_SUB;
  const size_t nr = (n2 + ((size_t)1 << bits) - 1) >> bits;
  if (n2 < OTP2_MIN_LITS || nr > OTP2_MAX_RANGES || !otp_plan(n2, ncls, p, tile_log2, xcd)) return false;
  p->bits = bits;
  p->nr = (u32)nr;
  p->ncounts = (size_t)p->nr * p->nblk;
  p->tiles2 = (u32)(pairs / OTP2_TILE + nr);
  p->ncounts2 = ((size_t)p->tiles2 << OTP2_SUB) + 1;
  return true;
}
// The same for a small formula: counted, scanned and placed in one launch
// without the pairs.  One workgroup walks the clauses twice where the tile and
// range kernels walk them once, on a workgroup per tile and per range of 1,024
// literals; what they lose are three launches.  So it is the faster way up to
// OT_ONE_LITS literals where there is one tile (its clauses are one workgroup's
// in either way), or where the clauses and occurrences are few for the number
// of ranges; past that, up to as many counters as the LDS holds, only for one
// tile of long clauses.  Whole calls, this against
// ranges: 500 variables, 16,000 clauses of 3 122 against 140 us; 1,000
// variables, 8,000 of 10 197 and 235, 16,000 of 10 225 and 215; 4,000
// variables, 4,000 of 3 118 and 117, 8,000 of 3 143 and 130, 4,000 of 100 620
// and 850; 5,000 variables, 6,500 of 3 130 and 124; 7,000 variables, 2,300 of 3
// 111 and 104, of 30 429 and 445, 2,000 of 1,000 3,540 and 4,480, 32,000 of 30
// 1,520 and 355.
template <bool TABLE>
__global__ void __launch_bounds__(OTP_TB) otp_one_k(DB db, u32 n2, u32* hist) {
  extern __shared__ u32 lc[];
  __shared__ u32 lw[OTP_TB / 64];
  for (u32 j = threadIdx.x; j < n2; j += OTP_TB) lc[j] = 0;
  __syncthreads();
  otp_tile(db, 0, db.ncls, [&](u32 l, u32) { atomicAdd(&lc[l], 1u); });
  __syncthreads();
  if (!TABLE) {
    for (u32 j = threadIdx.x; j < n2; j += OTP_TB) hist[j] = lc[j];
    return;
  }
  const u32 per = (n2 + OTP_TB - 1) / OTP_TB, j0 = threadIdx.x * per, j1 = min(n2, j0 + per);
  u32 s = 0, tot;
  for (u32 j = j0; j < j1; j++) s += lc[j];
  u32 pre = block_excl_scan_w<OTP_TB / 64>(s, lw, &tot);
  for (u32 j = j0; j < j1; j++) {
    const u32 v = lc[j];
    db.ot_off[j] = pre;
    db.ot_size[j] = v;
    hist[j] = v;
    lc[j] = pre;  // the list's cursor
    pre += v;
  }
  if (threadIdx.x == 0) db.ot_off[n2] = tot;
  __syncthreads();
  otp_tile(db, 0, db.ncls, [&](u32 l, u32 c) { db.ot_refs[atomicAdd(&lc[l], 1u)] = c; });
}
bool ot_one_fits(size_t n2, size_t ncls, size_t slots) {
  const size_t ranges = (n2 + 1023) >> 10;
  if (n2 > OT_ONE_LITS) return n2 <= OT_ONE_LITS_LONG && ncls <= OT_ONE_TILE && slots >= 16 * ncls;
  return ncls <= OT_ONE_TILE || (ncls * ranges <= OT_ONE_CLAUSES && slots * ranges <= OT_ONE_SLOTS);
}
void k_ot_one(const DB& db, u32 n2, bool table, u32* hist, Stream* st) {
  if (table) KLAUNCH_LDS(otp_one_k<true>, 1, OTP_TB, (size_t)n2 * 4, st, db, n2, hist);
  else KLAUNCH_LDS(otp_one_k<false>, 1, OTP_TB, (size_t)n2 * 4, st, db, n2, hist);
}
// counts: p.ncounts + 1 words; pairs: 8-byte aligned, two words per live
// occurrence (table) or one (hist only); tmp: scan_tmp_bytes(p.ncounts)
void k_ot_ranges2(const DB& db, const OtpPlan& p, u32 n2, u32* counts, u32* tb, u32* counts2, void* pairs,
                  void* pairs2, u32* hist, void* tmp, Stream* st) {
  const size_t lds_r = (size_t)p.nr * 4;
  const u32* total = counts + p.ncounts;
  KLAUNCH_LDS(otp_count_k, p.nblk, OTP_TB, lds_r, st, db, p.ct, p.bits, p.nr, p.nblk, p.xcd, counts);
  scan_u32(counts, counts, p.ncounts, counts + p.ncounts, tmp, st);
  KLAUNCH_LDS(otp_part_k<true>, p.nblk, OTP_TB, lds_r, st, db, p.ct, p.bits, p.nr, p.nblk, p.xcd, counts, pairs);
  KLAUNCH(otp2_tiles_k, 1, OTP2_MAX_RANGES, st, counts, p.nblk, p.nr, total, tb);
  KLAUNCH(otp2_count_k, p.tiles2, OTP_TB, st, counts, p.nblk, p.nr, total, tb, (const uint2*)pairs, counts2);
  scan_u32(counts2, counts2, p.ncounts2, nullptr, tmp, st);  // past the last tile's: the total
  KLAUNCH(otp2_part_k, p.tiles2, OTP_TB, st, counts, p.nblk, p.nr, total, tb, (const uint2*)pairs, counts2,
          (uint2*)pairs2);
  KLAUNCH(otp2_range_k, (n2 + (1u << OTP2_BITS) - 1) >> OTP2_BITS, OTP_RTB, st, db, n2, tb, counts2, total,
          (const uint2*)pairs2, hist);
}
void k_ot_ranges(const DB& db, const OtpPlan& p, u32 n2, u32* counts, void* pairs, bool table, u32* hist,
                 void* tmp, Stream* st) {
  const size_t lds_r = (size_t)p.nr * 4, lds_b = ((size_t)4 << p.bits);
  KLAUNCH_LDS(otp_count_k, p.nblk, OTP_TB, lds_r, st, db, p.ct, p.bits, p.nr, p.nblk, p.xcd, counts);
  scan_u32(counts, counts, p.ncounts, counts + p.ncounts, tmp, st);
  if (table) {
    KLAUNCH_LDS(otp_part_k<true>, p.nblk, OTP_TB, lds_r, st, db, p.ct, p.bits, p.nr, p.nblk, p.xcd, counts, pairs);
    KLAUNCH_LDS(otp_range_k<true>, p.nr, OTP_RTB, lds_b, st, db, p.bits, n2, p.nblk, counts, counts + p.ncounts, pairs,
                hist);
  } else {
    KLAUNCH_LDS(otp_part_k<false>, p.nblk, OTP_TB, lds_r, st, db, p.ct, p.bits, p.nr, p.nblk, p.xcd, counts,
                pairs);
    KLAUNCH_LDS(otp_range_k<false>, p.nr, OTP_RTB, lds_b, st, db, p.bits, n2, p.nblk, counts, counts + p.ncounts,
                pairs, hist);
  }
}

constexpr u32 SORT_SMALL = 16;
constexpr u32 SORT_BLOCK = 2048;
// wave-aggregated append: one atomic per wavefront per counter
__device__ inline void wave_append(bool pred, u32 val, u32* arr, u32* cnt) {
  const u64 mask = __ballot(pred);
  if (!mask) return;
  const int lane = threadIdx.x & 63;
  const int leader = __ffsll((unsigned long long)mask) - 1;
  u32 base = 0;
  if (lane == leader) base = atomicAdd(cnt, (u32)__popcll(mask));
  base = __shfl(base, leader, 64);
  if (pred) arr[base + __popcll(mask & ((1ull << lane) - 1))] = val;
}
// Lists of LO < len <= W entries (every length up to W when LO is 0)
// sorted by a group of W lanes: bitonic network over wave64 shuffles, keys
// in registers.  Also leaves in lsum[g] the sum of the clause sizes of such
// a list g (a bound for later stages: the lists of elected variables only
// shrink).  Returns the list's length.
template <u32 W, u32 LO>
__device__ inline u32 sort_group(const DB& db, u32 lit, bool valid, u32 j, u32 g, u32* lsum) {
  const u32 len0 = valid ? db.ot_size[lit] : 0;
  const bool mine = valid && len0 <= W && (LO == 0 || len0 > LO);
  const u32 small = mine ? len0 : 0;
  const u32 len = small >= 2 ? small : 0;
  u32* r = db.ot_refs + (small ? db.ot_off[lit] : 0);
  u64 a = ~0ull, b = ~0ull;
  u32 id = 0xFFFFFFFFu, sz = 0;
  if (j < small) {
    const SortKey k = make_key(db, r[j]);
    sz = k.size;
    if (len) {
      a = ((u64)k.size << 32) | k.lit0;
      b = ((u64)k.back << 32) | k.sig;
      id = k.id;
    }
  }
#pragma unroll
  for (u32 d = W / 2; d > 0; d >>= 1) sz += __shfl_xor(sz, d, 64);
  if (j == 0 && mine) lsum[g] = sz;
#pragma unroll
  for (u32 k = 2; k <= W; k <<= 1) {
#pragma unroll
    for (u32 d = k >> 1; d > 0; d >>= 1) {
      const u64 pa = __shfl_xor(a, d, 64), pb = __shfl_xor(b, d, 64);
      const u32 pid = __shfl_xor(id, d, 64);
      const bool mine_less = a != pa ? a < pa : (b != pb ? b < pb : id < pid);
      const bool up = (j & k) == 0, lower = (j & d) == 0;
      const bool keep_min = lower == up;
      if (keep_min != mine_less) {
        a = pa;
        b = pb;
        id = pid;
      }
    }
  }
  if (j < len) r[j] = id;
  return len0;
}
// Every list once by a 4-lane group (wavefront count and dependent loads
// per list, not the sorting, bound these passes): the lists of at most
// SORT_TINY entries, most of an election's, are sorted there; the others
// are flagged (fmid: up to SORT_SMALL entries, flong: beyond), compacted by
// scans and sorted by 16-lane groups, per workgroup or by the long-list
// merge.  (Tried: one 16-lane pass over every list, 1.09 ms on the
// heavy-tailed round's 6.1M lists; a worklist filled with one atomic per
// wavefront on a shared counter; a second pass over every list that skips
// the short ones; a bounded grid striding over the lists.)
// APPEND: the longer lists go straight to the collected ones (cnt[1] middle,
// cnt[0] long), one atomic per wavefront and kind: for up to
// SORT_APPEND_MAX lists that is cheaper than the flags' scans and packs.
constexpr u32 SORT_TINY = 4;
constexpr u32 SORT_APPEND_MAX = 1u << 17;
// list g of the elected variables: the positive and the negative one of
// variable g / 2
__device__ inline u32 list_lit(const u32* pv, u32 g) { return V2L(pv[g >> 1]) | (g & 1u); }
template <bool APPEND>
__global__ void sort_tiny_k(DB db, const u32* pv, u32 n, u32* lsum, u32* mid, u32* big, u32* cnt) {
  const u32 t = blockIdx.x * blockDim.x + threadIdx.x;
  const u32 g = t / SORT_TINY, j = t % SORT_TINY;
  const bool valid = g < n;
  const u32 len = sort_group<SORT_TINY, 0>(db, valid ? list_lit(pv, g) : 0u, valid, j, g, lsum);
  const bool one = valid && j == 0, m = one && len > SORT_TINY && len <= SORT_SMALL, l = one && len > SORT_SMALL;
  if (APPEND) {
    wave_append(m, g, mid, cnt + 1);
    wave_append(l, g, big, cnt);
  } else if (one) {  // flags
    mid[g] = m ? 1u : 0u;
    big[g] = l ? 1u : 0u;
  }
}
__global__ void sort_pack_k(const u32* fmid, const u32* flong, const u32* pmid, const u32* plong, u32 n, u32* mid,
                            u32* big) {
  const u32 g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= n) return;
  if (fmid[g]) mid[pmid[g]] = g;
  if (flong[g]) big[plong[g]] = g;
}
// the lists mid[0..*nmid), 16 lanes each; a bounded grid strides over them
// (the loop bound is the same for every lane of a wavefront)
__global__ void sort_mid_k(DB db, const u32* pv, const u32* mid, const u32* nmid, u32* lsum) {
  const u64 m = (u64)*nmid * SORT_SMALL;
  for (u64 base = (u64)blockIdx.x * blockDim.x; base < m; base += (u64)gridDim.x * blockDim.x) {
    const u64 t = base + threadIdx.x;
    const bool valid = t < m;
    const u32 g = valid ? mid[t / SORT_SMALL] : 0u;
    sort_group<SORT_SMALL, SORT_TINY>(db, valid ? list_lit(pv, g) : 0u, valid, (u32)(t % SORT_SMALL), g, lsum);
  }
}
// bitonic sort of one list per workgroup in LDS (16 < len <= SORT_BLOCK)
__device__ void sort_block_list(DB db, u32 lit, u32 g, u32* lsum, u64* ka, u64* kb, u32* kid, u32* lw) {
  const u32 len = db.ot_size[lit];
  u32* r = db.ot_refs + db.ot_off[lit];
  u32 N = 1;
  while (N < len) N <<= 1;
  u32 sz = 0;
  for (u32 i = threadIdx.x; i < N; i += blockDim.x) {
    if (i < len) {
      const SortKey k = make_key(db, r[i]);
      ka[i] = ((u64)k.size << 32) | k.lit0;
      kb[i] = ((u64)k.back << 32) | k.sig;
      kid[i] = k.id;
      sz += k.size;
    } else {
      ka[i] = ~0ull;
      kb[i] = ~0ull;
      kid[i] = 0xFFFFFFFFu;
    }
  }
  u32 tot;
  block_excl_scan(sz, lw, &tot);
  if (threadIdx.x == 0) lsum[g] = tot;
  for (u32 k = 2; k <= N; k <<= 1) {
    for (u32 j = k >> 1; j > 0; j >>= 1) {
      for (u32 i = threadIdx.x; i < N; i += blockDim.x) {
        const u32 ixj = i ^ j;
        if (ixj > i) {
          const bool up = (i & k) == 0;
          const u64 a0 = ka[i], a1 = ka[ixj], b0 = kb[i], b1 = kb[ixj];
          const u32 i0 = kid[i], i1 = kid[ixj];
          const bool gt = a0 != a1 ? a0 > a1 : (b0 != b1 ? b0 > b1 : i0 > i1);
          if (gt == up) {
            ka[i] = a1; ka[ixj] = a0;
            kb[i] = b1; kb[ixj] = b0;
            kid[i] = i1; kid[ixj] = i0;
          }
        }
      }
      __syncthreads();
    }
  }
  for (u32 i = threadIdx.x; i < len; i += blockDim.x) r[i] = kid[i];
}
// bottom-up merge sort of one long list by one thread (rare lists above
// SORT_BLOCK entries); 'scratch' has one slot per occurrence entry
__device__ void sort_large_list(DB db, u32 lit, u32 g, u32* scratch, u32* lsum) {
  const u32 len = db.ot_size[lit];
  u32* a = db.ot_refs + db.ot_off[lit];
  u64 sz = 0;
  for (u32 k = 0; k < len; k++) sz += csize(db, a[k]);
  lsum[g] = sz > 0xFFFFFFFFull ? 0xFFFFFFFFu : (u32)sz;
  u32* b = scratch + db.ot_off[lit];
  u32 *src = a, *dst = b;
  for (u32 w = 1; w < len; w <<= 1) {
    for (u32 lo = 0; lo < len; lo += 2 * w) {
      const u32 mid = lo + w < len ? lo + w : len;
      const u32 hi = lo + 2 * w < len ? lo + 2 * w : len;
      u32 p = lo, q = mid, o = lo;
      while (p < mid && q < hi) {
        if (key_less(make_key(db, src[q]), make_key(db, src[p]))) dst[o++] = src[q++];
        else dst[o++] = src[p++];
      }
      while (p < mid) dst[o++] = src[p++];
      while (q < hi) dst[o++] = src[q++];
    }
    u32* t = src; src = dst; dst = t;
  }
  if (src != a)
    for (u32 k = 0; k < len; k++) a[k] = src[k];
}
// the *nbig collected long lists (the count read on the device: a bounded
// grid strides over them, so the launch needs no host read of it)
__global__ void __launch_bounds__(256) sort_long_k(DB db, const u32* pv, const u32* big, const u32* nbig,
                                                   u32* scratch, u32* lsum) {
  __shared__ u64 ka[SORT_BLOCK];
  __shared__ u64 kb[SORT_BLOCK];
  __shared__ u32 kid[SORT_BLOCK];
  __shared__ u32 lw[NW];
  const u32 nb = *nbig;
  for (u32 b = blockIdx.x; b < nb; b += gridDim.x) {
    const u32 g = big[b], lit = list_lit(pv, g);
    if (db.ot_size[lit] <= SORT_BLOCK) sort_block_list(db, lit, g, lsum, ka, kb, kid, lw);
    else if (threadIdx.x == 0) sort_large_list(db, lit, g, scratch, lsum);
    __syncthreads();
  }
}
void k_sort_lists(const DB& db, const u32* pv, u32 nvars, u32* classes, u32* cnt, u32* scratch, u32* lsum,
                  void* tmp, Stream* st) {
  const u32 n = 2 * nvars;
  if (!n) return;
  u32* big = classes;           // lists longer than SORT_SMALL
  u32* mid = classes + n;       // lists of SORT_TINY < len <= SORT_SMALL
  const unsigned grid = grid_for((size_t)n * SORT_TINY, 256);
  if (n <= SORT_APPEND_MAX) {
    KLAUNCH(sort_tiny_k<true>, grid, 256, st, db, pv, n, lsum, mid, big, cnt);
  } else {
    u32* fmid = classes + 2 * (size_t)n;
    u32* flong = classes + 3 * (size_t)n;
    u32* pmid = classes + 4 * (size_t)n;
    u32* plong = classes + 5 * (size_t)n;
    KLAUNCH(sort_tiny_k<false>, grid, 256, st, db, pv, n, lsum, fmid, flong, cnt);
    scan_set(ScanSet{{flong, fmid}, {plong, pmid}, {cnt, cnt + 1}}, 2, n, tmp, st);
    KLAUNCH(sort_pack_k, grid_for(n, 256), 256, st, fmid, flong, pmid, plong, n, mid, big);
  }
  // the collected lists' launches read their counts on the device
  KLAUNCH(sort_mid_k, std::min(grid_for((size_t)n * SORT_SMALL, 256), 4096u), 256, st, db, pv, mid, cnt + 1, lsum);
  KLAUNCH(sort_long_k, std::min(n, 1024u), 256, st, db, pv, big, cnt, scratch, lsum);
}

// ---------------------------------------------------------------- BCP
// Kernels that walk the occurrence lists of a few literals (units): one
// row of workgroups per literal (blockIdx.y) strides over its list, so that
// a handful of hot literals (lists of 10^4-10^5 entries on heavy-tailed
// formulas) does not leave the device to one workgroup each.  The launcher
// aims at about 4096 workgroups in all and at most 65535 literals per
// launch (the grid's y extent).
template <class L>
void launch_per_literal(u32 n, L launch) {
  for (u32 c0 = 0; c0 < n; c0 += 65535) {
    const u32 m = std::min<u32>(n - c0, 65535);
    launch(dim3(std::max<u32>(1, std::min<u32>(64, 4096 / m)), m), c0);
  }
}
__device__ inline u32 list_lane() { return blockIdx.x * blockDim.x + threadIdx.x; }
__device__ inline u32 list_stride() { return gridDim.x * blockDim.x; }
__global__ void bcp_visit_k(DB db, const u32* front, u32* next, u32* nnext, u32* conflict) {
  const u32 t = front[blockIdx.y];
  const OLV ol = olist(db, FLIP(t));
  for (u32 i = list_lane(); i < ol.n; i += list_stride()) bcp_visit(db, ol.r[i], next, nnext, conflict);
}
void k_bcp_visit(const DB& db, const u32* front, u32 nfront, u32* next, u32* nnext, u32* conflict,
                 Stream* st) {
  launch_per_literal(nfront, [&](dim3 grid, u32 c0) {
    KLAUNCH(bcp_visit_k, grid, 256, st, db, front + c0, next, nnext, conflict);
  });
}
// Propagation level by level in one launch by one workgroup, as long as the
// levels stay narrow: trail[front..end) is the frontier, a wavefront takes a
// literal and its lanes the clauses of the list of its negation, the units
// found follow on the trail.  more (nullable): the frontier is what a launch of
// bcp_visit_k before this one appended, more[0] literals past 'end', unless
// more[1] says that it met a conflict.  Stops at the fixpoint, at a conflict
// (its level's units are not on the trail) or before a level that is not
// narrow, which bcp_visit_k spreads over the device; out: the trail's end, the
// conflict, the first literal not propagated yet.
//
// A wavefront spends a turn of 2.6 us, a chain of six dependent loads, on every
// list however short (1.4 us for each further 64 entries of a long one); a level
// by bcp_visit_k takes about 16 us with its read.  So a level is narrow by the
// turns that it takes, BCP_TURNS of them over the 16 wavefronts and BCP_LONG
// entries in one list.  Calls of 40 levels, all in one launch against a launch
// and a read each: 64 literals of 1, 16 and 64 entries 0.70, 0.84 and 1.08 ms
// against 0.87, 0.98 and 1.11; 128 literals 1.18, 1.47 and 1.95 against 1.01,
// 1.13 and 1.35; 1,024 literals of one entry 7.6 against 1.5; one list of 256,
// 1,024 and 16,384 entries 0.47, 1.09 and 14.8 against 0.86, 0.95 and 2.4.
constexpr u32 BCP_LONG = 512;
constexpr int BCP_T = 1024;
__global__ void __launch_bounds__(BCP_T) bcp_run_k(DB db, u32* trail, u32 front, u32 end, const u32* more, u32* out) {
  __shared__ u32 s_end, s_conflict, s_work[2];
  u32 conflict = 0;
  if (more) {
    conflict = more[1];
    if (!conflict) end += more[0];
  }
  if (threadIdx.x == 0) {
    s_end = end;
    s_conflict = 0;
    s_work[0] = s_work[1] = 0;
  }
  __syncthreads();
  for (u32 level = 0; !conflict && front < end && end - front <= BCP_TURNS; level++) {
    u32 w = 0;
    for (u32 i = front + threadIdx.x; i < end; i += BCP_T) {
      const u32 n = db.ot_size[FLIP(trail[i])];
      w += n > BCP_LONG ? BCP_TURNS + 1 : max(1u, (n + 63) / 64);
    }
    if (w) atomicAdd(&s_work[level & 1], w);
    __syncthreads();
    if (s_work[level & 1] > BCP_TURNS) break;
    if (threadIdx.x == 0) s_work[(level + 1) & 1] = 0;
    for (u32 i = front + threadIdx.x / 64; i < end; i += BCP_T / 64) {
      const OLV ol = olist(db, FLIP(trail[i]));
      for (u32 j = threadIdx.x & 63; j < ol.n; j += 64) bcp_visit(db, ol.r[j], trail, &s_end, &s_conflict);
    }
    __syncthreads();
    conflict = s_conflict;
    if (conflict) break;
    front = end;
    end = s_end;
    __syncthreads();  // every thread has read them before the next level appends
  }
  if (threadIdx.x == 0) {
    out[0] = end;
    out[1] = conflict;
    out[2] = front;
  }
}
void k_bcp_run(const DB& db, u32* trail, u32 front, u32 end, const u32* more, u32* out, Stream* st) {
  KLAUNCH(bcp_run_k, 1, BCP_T, st, db, trail, front, end, more, out);
}
__global__ void bcp_mark_k(DB db, const u32* lits, u8* mark) {
  const u32 t = lits[blockIdx.y];
  for (u32 q = 0; q < 2; q++) {
    const OLV ol = olist(db, t ^ q);
    for (u32 i = list_lane(); i < ol.n; i += list_stride()) mark[ol.r[i]] = 1;
  }
}
void k_bcp_mark(const DB& db, const u32* lits, u32 n, u8* mark, Stream* st) {
  launch_per_literal(n, [&](dim3 grid, u32 c0) { KLAUNCH(bcp_mark_k, grid, 256, st, db, lits + c0, mark); });
}
// mark: per handle
__global__ void bcp_clean_k(DB db, u8* mark) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= db.ncls) return;
  const u32 c = db.c_off[i];
  if (!mark[c]) return;
  mark[c] = 0;
  bcp_clean(db, c);
}
void k_bcp_clean(const DB& db, u8* mark, Stream* st) {
  if (!db.ncls) return;
  KLAUNCH(bcp_clean_k, grid_for(db.ncls, 256), 256, st, db, mark);
}
__global__ void clear_lists_k(DB db, const u32* lits, u32 n) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const u32 t = lits[i];
  db.ot_size[t] = 0;
  db.ot_size[FLIP(t)] = 0;
}
void k_clear_lists(const DB& db, const u32* lits, u32 n, Stream* st) {
  if (!n) return;
  KLAUNCH(clear_lists_k, grid_for(n, 256), 256, st, db, lits, n);
}
__global__ void set_vstate_k(DB db, const u32* lits, u32 n, u8 state) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) db.vstate[ABS(lits[i])] = state;
}
void k_set_vstate(const DB& db, const u32* lits, u32 n, u8 state, Stream* st) {
  if (!n) return;
  KLAUNCH(set_vstate_k, grid_for(n, 256), 256, st, db, lits, n, state);
}

// ---------------------------------------------------------------- LCVE
__device__ unsigned long long lcve_classify_var(const DB& db, const LcveArgs& a, u32 v, u32& top);
__device__ inline unsigned long long wave_min64(unsigned long long x) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const unsigned long long y = __shfl_xor(x, d, 64);
    x = y < x ? y : x;
  }
  return x;
}
// the hard-break key is a minimum over the grid: per lane over a strided
// range of variables, then over the workgroup, then one atomic per
// workgroup into a bounded grid (one atomic per wavefront over 10M
// variables serialised 1 ms on the one word)
__global__ void lcve_classify_k(DB db, LcveArgs a) {
  __shared__ unsigned long long wmin[ST / 64];
  __shared__ u32 wmax[ST / 64];
  unsigned long long hk = ~0ull;
  u32 top = 0;
  for (u32 v = blockIdx.x * blockDim.x + threadIdx.x + 1; v <= db.nvars; v += gridDim.x * blockDim.x) {
    const unsigned long long k = lcve_classify_var(db, a, v, top);
    hk = k < hk ? k : hk;
  }
  hk = wave_min64(hk);
  top = wave_max(top);
  if ((threadIdx.x & 63) == 0) {
    wmin[threadIdx.x >> 6] = hk;
    wmax[threadIdx.x >> 6] = top;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (u32 w = 1; w < ST / 64; w++) {
      hk = wmin[w] < hk ? wmin[w] : hk;
      top = max(top, wmax[w]);
    }
    if (hk != ~0ull) at_min64(a.hard, hk);
    if (top) atomicMax(&a.top[blockIdx.x % LCVE_TOPS], top);
  }
}
__device__ unsigned long long lcve_classify_var(const DB& db, const LcveArgs& a, u32 v, u32& top) {
  const u32 ps = a.hist[V2L(v)], ns = a.hist[V2L(v) | 1];
  const u32 score = ps * ns;  // 32-bit product as in the reference
  a.score[v] = score;
  const bool cand = !db.assumed[v] && !db.vstate[v] && (ps || ns);
  // break rules (lcve.cpp:61-66; the GPU build's electionsmax, lcve.cu:94)
  const bool brk = (db.ot_size[V2L(v)] >= a.pt && db.ot_size[V2L(v) | 1] >= a.nt) || ps > a.max_occurs ||
                   ns > a.max_occurs;
  // a breaker that no neighbour can freeze (the freeze rule spares variables
  // at or above both temperatures) ends the election wherever it stands
  const bool hard = brk && ps >= a.pt && ns >= a.nt;
  u8 f = cand ? (brk ? 3 : 1) : 0;
  if (f == 1 && a.clause_max != 0xFFFFFFFFu && lcve_oversize(db, v, a.clause_max)) f = 4;
  a.cflag[v] = f;
  if (f) top = max(top, score);
  return cand && hard ? ((unsigned long long)score << 32) | v : ~0ull;
}
__global__ void lcve_clear_k(LcveArgs a) {
  a.top[threadIdx.x] = 0;
  if (threadIdx.x == 0) *a.hard = ~0ull;
}
void k_lcve_classify(const DB& db, const LcveArgs& a, Stream* st) {
  KLAUNCH(lcve_clear_k, 1, LCVE_TOPS, st, a);
  KLAUNCH(lcve_classify_k, std::min(grid_for(db.nvars, ST), 2048u), ST, st, db, a);
}
__global__ void lcve_flag_k(DB db, LcveArgs a, u32* flag, u32* pos) {
  const u32 v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v > db.nvars) return;
  pos[v] = NOPOS;
  u32 f = 0;
  if (v && a.cflag[v]) f = (((u64)a.score[v] << 32) | v) < *a.hard;
  flag[v] = f;
}
__global__ void lcve_pack_k(DB db, LcveArgs a, const u32* flag, const u32* pos, u32* cand, u32* key) {
  const u32 v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v > db.nvars || !v) return;
  if (!a.cflag[v] || !((((u64)a.score[v] << 32) | v) < *a.hard)) return;
  const u32 i = pos[v];
  cand[i] = v;
  key[i] = a.score[v];
}
void k_lcve_select(const DB& db, const LcveArgs& a, u32* flag_tmp, u32* cand, u32* key, u32* pos, u32* ncand,
                   void* tmp, Stream* st) {
  const size_t n = (size_t)db.nvars + 1;
  KLAUNCH(lcve_flag_k, grid_for(n, 256), 256, st, db, a, flag_tmp, pos);
  scan_u32(flag_tmp, flag_tmp, n, ncand, tmp, st);
  KLAUNCH(lcve_pack_k, grid_for(n, 256), 256, st, db, a, flag_tmp, flag_tmp, cand, key);
}
// The state of an election before its first step: each candidate's packed
// position and state (undecided, or decided and not elected for the ones
// passed over) and the counters (sc: [1] the break position, [3..6] and
// [12..14] the passes' counts, [24..25] the list sort's), in one launch.  The positions of variables
// that are no candidates are NOPOS from lcve_flag_k.
__global__ void mis_init_k(const u32* cand, u32 n, const u8* cflag, bool reject, u32* pos, u32* state, u32* sc) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    sc[1] = n;
    sc[3] = 0;
    for (u32 q = 0; q < 3; q++) sc[4 + q] = 0, sc[12 + q] = 0;
    sc[24] = sc[25] = 0;
  }
  if (i >= n) return;
  const u32 v = cand[i], st = reject && cflag[v] == 4 ? 2u : 0u;
  state[i] = st;
  pos[v] = (i << 2) | st;
}
void k_mis_init(const u32* cand, u32 n, const u8* cflag, bool reject, u32* pos, u32* state, u32* sc, Stream* st) {
  KLAUNCH(mis_init_k, std::max(1u, grid_for(n, 256)), 256, st, cand, n, cflag, reject, pos, state, sc);
}
// One election step by a group of G lanes per candidate (G a power of two,
// groups aligned in the wavefront): the lanes share out the entries of the
// candidate's two lists (positive, then negative: one combined index) and
// combine their findings, an elected earlier neighbour anywhere freezes
// the candidate, else the earliest entry holding an undecided earlier
// neighbour is its blocker's entry.  The outcome is the one-lane scan's
// (mis_step); G lanes keep G chains of loads in flight per candidate.
// The blocker and the entry to go on from are the same in every lane of the
// group and stay in registers (b, r) while the candidate is tried again.
// Returns 1 if the candidate stays undecided (in every lane of the group).
template <u32 G>
__device__ inline u32 mis_try(const DB& db, u32 i, u32 v, u32* pw, u32* state, u32& b, u32& r) {
  const int lane = threadIdx.x & 63, lead = lane & ~(int)(G - 1), j = lane - lead;
  if (b != NOPOS) {
    u32 sb = j == 0 ? at_load(&state[b]) : 0u;
    sb = __shfl(sb, lead, 64);
    if (sb == 0) return 1;
    if (sb == 1) {
      if (j == 0) mis_decide(state, pw, i, v, 2);
      return 0;
    }
  }
  const OLV o0 = olist(db, V2L(v)), o1 = olist(db, V2L(v) | 1);
  const u32 n0 = o0.n, ntot = o0.n + o1.n;
  u32 first = NOPOS, bpos = NOPOS;  // this lane's earliest entry with an undecided earlier neighbour
  bool frozen = false;
  for (u32 e = r + j; e < ntot && !frozen; e += G) {
    const u32 c = e < n0 ? o0.r[e] : o1.r[e - n0];
    const u32 h = db.lits[c];
    if (st_deleted(hdr_flags(h))) continue;
    const u32* l = db.lits + c + CL_HDR;
    const u32 n = hdr_size(h);
    for (u32 q = 0; q < n && !frozen; q += 4) {
      u32 u[4], w[4];
#pragma unroll
      for (u32 k = 0; k < 4; k++) u[k] = q + k < n ? ABS(l[q + k]) : v;
#pragma unroll
      for (u32 k = 0; k < 4; k++) w[k] = u[k] != v ? at_load(&pw[u[k]]) : NOPOS;
#pragma unroll
      for (u32 k = 0; k < 4; k++) {
        const u32 pu = w[k] >> 2;  // NOPOS: past every candidate
        if (pu >= i) continue;
        const u32 su = w[k] & 3u;
        if (su == 1) frozen = true;
        if (su == 0 && first == NOPOS) first = e, bpos = pu;
      }
    }
  }
  u32 fz = frozen ? 1u : 0u;
  u64 m = ((u64)first << 32) | bpos;
#pragma unroll
  for (u32 d = 1; d < G; d <<= 1) {
    fz |= __shfl_xor(fz, d, 64);
    const u64 o = __shfl_xor(m, d, 64);
    m = o < m ? o : m;
  }
  if (fz) {
    if (j == 0) mis_decide(state, pw, i, v, 2);
    return 0;
  }
  r = (u32)(m >> 32);
  b = (u32)m;
  if (r != NOPOS) return 1;
  if (j == 0) mis_decide(state, pw, i, v, 1);
  return 0;
}
// Candidate i (each group its own) until it is decided, at most 'tries'
// times: a candidate's blocker is decided by another wavefront of the same
// launch as a rule, so waiting a little costs a poll of the blocker's state
// where another pass costs a launch, the list entries again and a worklist
// append.  No try waits for anything: one that stays undecided leaves its
// blocker and entry in blk / resume and is appended to 'next'.
template <u32 G>
__device__ inline void mis_run(const DB& db, u32 i, bool valid, bool fresh, const u32* cand, u32* pos, u32* state,
                               u32* blk, u32* resume, u32* next, u32* nnext, u32 tries) {
  const bool lead = (threadIdx.x & (G - 1)) == 0;
  bool undecided = valid && state[i] == 0;  // set before this launch: nothing decides i but this group
  u32 v = 0, b = NOPOS, r = 0;
  if (undecided) {
    v = cand[i];
    if (!fresh) b = blk[i], r = resume[i];
  }
  for (u32 t = 0; t < tries && __any(undecided); t++) {
    if (t) __builtin_amdgcn_s_sleep(1);
    if (undecided) undecided = mis_try<G>(db, i, v, pos, state, b, r) != 0;
  }
  if (undecided && lead) {
    blk[i] = b;
    resume[i] = r;
  }
  wave_append(undecided && lead, i, next, nnext);
}

// the first pass, over all candidates; the ones still undecided are appended
// to 'next'.  The launch reserves LDS per one-wavefront workgroup only to
// bound occupancy (option "mislds"; 20 KiB leaves 2 wavefronts per SIMD:
// Tseitin round 0 / 20 / 40 KiB -> mis_step_k 3.34 / 2.76 / 3.18 ms)
template <u32 G>
__global__ void mis_step_k(DB db, const u32* cand, u32 n, const u32* n_dev, u32* pos, u32* state, u32* blk, u32* resume,
                           u32* next, u32* nnext, u32 tries) {
  if (n_dev) n = *n_dev;
  const u64 t = (u64)blockIdx.x * blockDim.x + threadIdx.x;
  const u32 q = (u32)(t / G);
  mis_run<G>(db, q, q < n, true, cand, pos, state, blk, resume, next, nnext, tries);
}
// A worklist pass whose length is read on the device (n_in): a bounded grid
// strides over the list, so several passes are queued without a host read;
// passes over an empty list return at once.  iters counts the non-empty passes.
// zero: the counter the next pass appends to (the input counter of the
// pass before this one, so nothing reads it any more), cleared here instead
// of by a launch of its own before every pass
template <u32 G>
__global__ void mis_step_dev_k(DB db, const u32* cand, const u32* idx, const u32* n_in, u32* pos, u32* state,
                               u32* blk, u32* resume, u32* next, u32* nnext, u32* iters, u32* zero, u32 tries) {
  const u32 n = *n_in;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *zero = 0;
    if (n) atomicAdd(iters, 1u);
  }
  const u64 m = (u64)n * G;
  for (u64 base = (u64)blockIdx.x * blockDim.x; base < m; base += (u64)gridDim.x * blockDim.x) {  // wave-uniform
    const u32 q = (u32)((base + threadIdx.x) / G);
    mis_run<G>(db, q < n ? idx[q] : 0u, q < n, false, cand, pos, state, blk, resume, next, nnext, tries);
  }
}
#define MIS_LANES(G, call) \
  switch (G) {             \
    case 2: call(2); break; \
    case 4: call(4); break; \
    case 8: call(8); break; \
    case 16: call(16); break; \
    default: call(1); break; \
  }
// tries per candidate and pass: 1 / 4 / 16 / 64 tries took the election's
// passes on 10M heavy-tailed variables from 3.17 + 0.62 to 3.08 + 0.05 ms
// (4 and more alike), and a 20,000-variable call from 2.43 (1) to 1.63 (4)
// and 1.58 ms (16)
constexpr u32 MIS_TRIES = 32;
// lanes per candidate by their number: up to 16 while all the groups fit
// twice the wavefronts in flight (16 per CU at 10 KiB of LDS each; once, twice
// and four times measured alike from 301 to 340,000 clauses).  A small
// formula's step is a chain of dependent loads per list entry, which 16
// lanes walk 16 entries at a time: with one lane the two first passes of the
// 20,000-variable round took 89 us, with 16 lanes 98 us with all tries but
// the last in them.
u32 mis_lanes_for(u32 n) {
  constexpr u64 in_flight = 256 * 16 * 64;
  u32 g = 16;
  while (g > 1 && (u64)n * g > 2 * in_flight) g >>= 1;
  return g;
}
void k_mis_step(const DB& db, const u32* cand, u32 n, const u32* n_dev, u32* pos, u32* state, u32* blk, u32* resume,
                u32* next, u32* nnext, u32 lds, u32 lanes, Stream* st) {
  if (!n) return;
#define MIS_FIRST(G) \
  KLAUNCH_LDS(mis_step_k<G>, grid_for((size_t)n * G, 64), 64, lds, st, db, cand, n, n_dev, pos, state, blk, resume, \
              next, nnext, MIS_TRIES)
  MIS_LANES(lanes, MIS_FIRST)
#undef MIS_FIRST
}
void k_mis_step_dev(const DB& db, const u32* cand, const u32* idx, const u32* n_in, u32 n_bound, u32* pos,
                    u32* state, u32* blk, u32* resume, u32* next, u32* nnext, u32* iters, u32* zero, u32 lds,
                    u32 lanes, Stream* st) {
  if (!n_bound) return;
#define MIS_DEV(G)                                                                                           \
  KLAUNCH_LDS(mis_step_dev_k<G>, std::min(grid_for((size_t)n_bound * G, 64), 2048u), 64, lds, st, db, cand, idx, \
              n_in, pos, state, blk, resume, next, nnext, iters, zero, MIS_TRIES)
  MIS_LANES(lanes, MIS_DEV)
#undef MIS_DEV
}
#undef MIS_LANES
__global__ void mis_break_k(const u32* cand, u32 n, const u8* cflag, const u32* state, u32* brk) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && state[i] == 1 && cflag[cand[i]] == 3) atomicMin(brk, i);
}
void k_mis_break(const u32* cand, u32 n, const u8* cflag, const u32* state, u32* brk, Stream* st) {
  if (!n) return;
  KLAUNCH(mis_break_k, grid_for(n, 256), 256, st, cand, n, cflag, state, brk);
}
__global__ void mis_flag_k(const u32* state, u32 n, const u32* brk, u32* flag) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flag[i] = (state[i] == 1 && i < *brk) ? 1u : 0u;
}
// entries (nullable): also sums the elected lists' entries (SUB's room), which
// the read of the number of elected variables brings along
__global__ void __launch_bounds__(256) mis_pack_k(DB db, const u32* cand, const u32* state, u32 n, const u32* brk,
                                                  const u32* pos, u32* out, u32* entries) {
  u32 w = 0;
  const u32 b = *brk;
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    if (state[i] == 1 && i < b) {
      const u32 v = cand[i];
      out[pos[i]] = v;
      if (entries) w += db.ot_size[V2L(v)] + db.ot_size[V2L(v) | 1];
    }
  if (!entries) return;
  __shared__ u32 lw[256 / 64];
  u32 tot;
  block_excl_scan_w<256 / 64>(w, lw, &tot);
  if (threadIdx.x == 0 && tot) atomicAdd(entries, tot);
}
void k_mis_collect(const DB& db, const u32* cand, u32 n, const u32* state, u32* flag_tmp, u32* out, u32* sc,
                   bool entries, void* tmp, Stream* st) {
  if (!n) {
    fill_u32(sc, 0, 1, st);
    return;
  }
  KLAUNCH(mis_flag_k, grid_for(n, 256), 256, st, state, n, sc + 1, flag_tmp);
  scan_u32(flag_tmp, flag_tmp, n, sc, tmp, st);
  KLAUNCH(mis_pack_k, entries ? std::min(grid_for(n, 256), RED_BLOCKS) : grid_for(n, 256), 256, st, db, cand, state, n,
          sc + 1, flag_tmp, out, entries ? sc + 3 : nullptr);
}

// Small formulas (up to LCVE_SMALL variables): everything around the election
// passes in one workgroup and one launch on either side of them, with the
// number of candidates kept on the device.  Classification, selection, sort
// and the initial states were eight launches and a read of the candidates'
// number, break, flags, scan and collection four more, 3-5 us each in a round
// whose kernels run as long.  With the table above, a call takes 0.82 ms
// instead of 0.96 at 301 variables (106 launches instead of 154) and 3.17
// instead of 3.35 at 5,000.
static_assert(LCVE_SMALL == SO_MAX, "one item per variable");
__global__ void __launch_bounds__(SO_T) lcve_small_k(DB db, LcveArgs a, bool reject, u32* pos, u32* cand, u32* state,
                                                     u32* sc) {
  constexpr int IPT = SO_IPT, W = SO_T / 64;
  __shared__ u32 sk[lpad(SO_MAX)];
  __shared__ uint16_t si[lpad(SO_MAX)];
  __shared__ u32 lw[W], wmax[W];
  __shared__ u64 lw64[W], wmin[W];
  unsigned long long hk = ~0ull;
  u32 top = 0;
  for (u32 v = threadIdx.x; v <= db.nvars; v += SO_T) {
    pos[v] = NOPOS;
    if (!v) continue;
    const unsigned long long k = lcve_classify_var(db, a, v, top);
    hk = k < hk ? k : hk;
  }
  hk = wave_min64(hk);
  top = wave_max(top);
  if ((threadIdx.x & 63) == 0) {
    wmin[threadIdx.x >> 6] = hk;
    wmax[threadIdx.x >> 6] = top;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < W; w++) {
    hk = wmin[w] < hk ? wmin[w] : hk;
    top = max(top, wmax[w]);
  }
  // the candidates before the hard breaker, in variable order
  const u32 j0 = threadIdx.x * IPT;
  u32 k[IPT], id[IPT], d[IPT], dst[IPT], keep = 0, n;
#pragma unroll
  for (int i = 0; i < IPT; i++) {
    const u32 v = j0 + i + 1;
    k[i] = 0;
    if (v <= db.nvars && a.cflag[v]) {
      k[i] = a.score[v];
      if ((((u64)k[i] << 32) | v) < hk) keep |= 1u << i;
    }
  }
  u32 at = block_excl_scan_w<W>(__popc(keep), lw, &n);
#pragma unroll
  for (int i = 0; i < IPT; i++)
    if (keep >> i & 1) {
      sk[lpad(at)] = k[i];
      si[lpad(at++)] = (uint16_t)(j0 + i);
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < IPT; i++) {  // slots past the candidates stay behind them
    const bool in = j0 + i < n;
    k[i] = in ? sk[lpad(j0 + i)] : 0xFFFFFFFFu;
    id[i] = in ? si[lpad(j0 + i)] : 0u;
  }
  __syncthreads();
  const u32 most = min((u32)(hk >> 32), top);
  const int bits = most ? 32 - __clz(most) : 0;
  for (int bit = 0; bit < bits; bit += 2) {
#pragma unroll
    for (int i = 0; i < IPT; i++) d[i] = (k[i] >> bit) & (bit + 1 < bits ? 3u : 1u);
    split4<SO_T, IPT>(d, dst, lw64);
#pragma unroll
    for (int i = 0; i < IPT; i++) {
      sk[lpad(dst[i])] = k[i];
      si[lpad(dst[i])] = (uint16_t)id[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IPT; i++) {
      k[i] = sk[lpad(j0 + i)];
      id[i] = si[lpad(j0 + i)];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < IPT; i++) {
    const u32 j = j0 + i;
    if (j >= n) continue;
    const u32 v = id[i] + 1, st = reject && a.cflag[v] == 4 ? 2u : 0u;
    cand[j] = v;
    state[j] = st;
    pos[v] = (j << 2) | st;
  }
  if (threadIdx.x == 0) {  // as mis_init_k, and the candidates
    sc[1] = sc[2] = n;
    sc[3] = 0;
    for (u32 q = 0; q < 3; q++) sc[4 + q] = 0, sc[12 + q] = 0;
    sc[24] = sc[25] = 0;
  }
}
void k_lcve_small(const DB& db, const LcveArgs& a, bool reject, u32* pos, u32* cand, u32* state, u32* sc, Stream* st) {
  KLAUNCH(lcve_small_k, 1, SO_T, st, db, a, reject, pos, cand, state, sc);
}
__global__ void __launch_bounds__(SO_T) collect_small_k(DB db, const u32* cand, const u8* cflag, const u32* state,
                                                        u32* out, u32* sc) {
  constexpr int IPT = SO_IPT, W = SO_T / 64;
  __shared__ u32 lw[W];
  __shared__ u32 brk;
  const u32 n = sc[2], j0 = threadIdx.x * IPT;
  if (threadIdx.x == 0) brk = n;
  __syncthreads();
  u32 v[IPT], el = 0;
#pragma unroll
  for (int i = 0; i < IPT; i++) {
    v[i] = 0;
    if (j0 + i >= n || state[j0 + i] != 1) continue;
    v[i] = cand[j0 + i];
    el |= 1u << i;
    if (cflag[v[i]] == 3) atomicMin(&brk, j0 + i);
  }
  __syncthreads();
  const u32 b = brk;
#pragma unroll
  for (int i = 0; i < IPT; i++)
    if (j0 + i >= b) el &= ~(1u << i);
  u32 tot, entries, w = 0;
  u32 at = block_excl_scan_w<W>(__popc(el), lw, &tot);
#pragma unroll
  for (int i = 0; i < IPT; i++)
    if (el >> i & 1) {
      out[at++] = v[i];
      w += db.ot_size[V2L(v[i])] + db.ot_size[V2L(v[i]) | 1];
    }
  block_excl_scan_w<W>(w, lw, &entries);
  if (threadIdx.x == 0) {
    sc[0] = tot;
    sc[1] = b;
    sc[3] = entries;
  }
}
void k_collect_small(const DB& db, const u32* cand, const u8* cflag, const u32* state, u32* out, u32* sc, Stream* st) {
  KLAUNCH(collect_small_k, 1, SO_T, st, db, cand, cflag, state, out, sc);
}

// ---------------------------------------------------------------- per elected variable
constexpr int VB = 64;  // one wavefront per workgroup for divergent per-variable work

__global__ void list_sizes_k(DB db, const u32* pv, u32 n, u32 extra, u32* out) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) out[k] = db.ot_size[V2L(pv[k])] + db.ot_size[V2L(pv[k]) | 1] + extra;
}
void k_list_sizes(const DB& db, const u32* pv, u32 n, u32 extra, u32* out, Stream* st) {
  if (!n) return;
  KLAUNCH(list_sizes_k, grid_for(n, 256), 256, st, db, pv, n, extra, out);
}
__global__ void sub_snapshot_k(DB db, const u32* pv, u32 n, SubSnap s) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) sub_snapshot_var(db, pv[k], k, s);
}
void k_sub_snapshot(const DB& db, const u32* pv, u32 n, const SubSnap& s, Stream* st) {
  if (!n) return;
  KLAUNCH(sub_snapshot_k, grid_for(n, VB), VB, st, db, pv, n, s);
}
__global__ void sub_restore_k(DB db, const u32* pv, const u32* idx, u32 n, SubSnap s) {
  const u32 t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) sub_restore_var(db, pv[idx[t]], idx[t], s);
}
void k_sub_restore(const DB& db, const u32* pv, const u32* idx, u32 n, const SubSnap& s, Stream* st) {
  if (!n) return;
  KLAUNCH(sub_restore_k, grid_for(n, VB), VB, st, db, pv, idx, n, s);
}
// one workgroup per unit change (elected index, literal, pass): flag the
// owners of the clauses in the literal's list that come after the deriving
// variable and last ran no later than that pass
// one row of workgroups per change (its unit's list: launch_per_literal)
__global__ void sub_affected_k(DB db, SubSnap s, const u32* ch, const u32* lastrun, u32* aff) {
  const u64 c = 3 * (u64)blockIdx.y;
  const u32 k_unit = ch[c], u = ch[c + 1], pass = ch[c + 2];
  const OLV ol = olist(db, u);
  for (u32 i = list_lane(); i < ol.n; i += list_stride()) {
    const u32 o = sub_affected_owner(s, ol.r[i], k_unit, lastrun, pass);
    if (o != NOPOS) aff[o] = 1;
  }
}
void k_sub_affected(const DB& db, const SubSnap& s, const u32* changes, u32 nch, const u32* lastrun, u32* aff,
                    Stream* st) {
  launch_per_literal(nch, [&](dim3 grid, u32 c0) {
    KLAUNCH(sub_affected_k, grid, 256, st, db, s, changes + 3 * (size_t)c0, lastrun, aff);
  });
}
__global__ void set_at_k(u32* dst, const u32* idx, u32 n, u32 value) {
  const u32 t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) dst[idx[t]] = value;
}
void k_set_at(u32* dst, const u32* idx, u32 n, u32 value, Stream* st) {
  if (!n) return;
  KLAUNCH(set_at_k, grid_for(n, 256), 256, st, dst, idx, n, value);
}
// triples (variable, elected index, literal): ust[variable] / ulit[variable]
__global__ void set_vis_k(u32* ust, u32* ulit, const u32* e, u32 n) {
  const u32 t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  ust[e[3 * t]] = e[3 * t + 1];
  ulit[e[3 * t]] = e[3 * t + 2];
}
void k_set_vis(u32* ust, u32* ulit, const u32* entries, u32 n, Stream* st) {
  if (!n) return;
  KLAUNCH(set_vis_k, grid_for(n, 256), 256, st, ust, ulit, entries, n);
}
__global__ void pack_flags_k(const u32* flags, const u32* pos, u32 n, u32* out) {
  const u32 t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n && flags[t]) out[pos[t]] = t;
}
void k_pack_flags(const u32* flags, u32 n, u32* pos, u32* out, u32* count, void* tmp, Stream* st) {
  if (!n) {
    fill_u32(count, 0, 1, st);
    return;
  }
  scan_u32(flags, pos, n, count, tmp, st);
  KLAUNCH(pack_flags_k, grid_for(n, 256), 256, st, flags, pos, n, out);
}
__global__ void oblivion_k(DB db, const u32* lits) {
  const u32 t = lits[blockIdx.y];
  const OLV ol = olist(db, t);
  for (u32 i = list_lane(); i < ol.n; i += list_stride()) set_deleted(db, ol.r[i]);
}
void k_oblivion(const DB& db, const u32* lits, u32 n, Stream* st) {
  launch_per_literal(n, [&](dim3 grid, u32 c0) { KLAUNCH(oblivion_k, grid, 256, st, db, lits + c0); });
}
// Per-variable searches over a variable's own two occurrence lists (SUB,
// the VE decisions that are not settled by the gate checks) re-read those
// lists all along.  Each variable copies them (lview_words / sview_words
// words) into LDS and works there.  A workgroup of LV_WAVES wavefronts has
// LV_WAVE_LDS bytes (cap words) for each.  A wavefront's share is divided
// among the variables of one size class: class q < LV_BIG gives 32 >> q of
// them 2 << q lanes and cap / (32 >> q) words each.  Lists larger than that
// (class LV_BIG) take the whole workgroup's LDS, one variable at a time on
// its first wavefront, and the last class, larger still, works on the pool,
// 64 variables to a wavefront.  A wavefront thus runs variables of like size,
// the largest first, and no lane that reads the pool holds up lanes that work
// in LDS.
//
// The kernels are bound by chains of dependent LDS reads, so by how many
// wavefronts hide each other's: with 20 KiB to each (8 on a CU) the decisions
// and SUB of a round took 0.90 + 0.55 ms on the circuit of 2M gates, 0.43 +
// 0.27 ms on 77,777 variables (three rounds) and 1.04 + 0.77 ms on 100,000
// gates (five); with 5 KiB (registers allow 24 on a CU) 0.49 + 0.32, 0.24 +
// 0.16 and 0.60 + 0.50 ms.  3 and 4 KiB are within 10 % of it either way, and
// with 4 KiB the largest lists that fit would be smaller.
//
// work: LV_WORK_HDR words (the first positions of the keys 0..8 in the
// placed order), then n elected indices.  The key of a variable of class c
// is LV_CLASSES - 1 - c (the largest lists first); VE execution gives the
// variables it keeps key LV_CLASSES.  place() orders them; within a class
// SUB and the VE decisions take the longest lists first (lv_fine), so that
// the variables of a wavefront have similar work (without it ve_decide_k
// took 1.11 instead of 0.89 ms on the 2M-gate circuit and sub_k 2.32 instead
// of 2.06 ms on 10M heavy-tailed variables).
constexpr u32 LV_CLASSES = 8, LV_BIG = LV_CLASSES - 2;
constexpr u32 LV_WAVES = 4, LV_WAVE_LDS = 5120, LV_LDS = LV_WAVES * LV_WAVE_LDS, LV_CAP = LV_WAVE_LDS / 4;
constexpr u32 LV_WORK_HDR = 32;
constexpr int LV_KEY_BITS = 4;
static_assert(LV_CLASSES + 1 <= LV_WORK_HDR && LV_CLASSES < (1u << LV_KEY_BITS) && LV_CLASSES == LV_KEPT,
              "class keys");
__device__ inline u32 lv_class(u64 need) {
  u32 q = 0;
  while (q < LV_BIG && need * (32u >> q) > LV_CAP) q++;
  return q == LV_BIG && need > LV_WAVES * LV_CAP ? LV_CLASSES - 1 : q;
}
__device__ inline u32 lv_class_lanes(u32 q) { return q < LV_BIG ? 32u >> q : 64u; }
// list occurrences as a descending 5-bit code: exact below 16, then four
// steps per power of two up to 256
constexpr int LV_FINE_BITS = 5;
__device__ inline u32 lv_fine(u32 w) {
  if (w < 16) return 31 - w;
  const u32 e = 31 - __clz(w);
  return 31 - min(31u, 16 + (e - 4) * 4 + ((w >> (e - 2)) & 3u));
}
// grid-stride over the chunks of all classes, a wavefront to a chunk;
// f(k, w, slice, gl, G) runs elected index k with the LDS words
// [w, w + slice) (w null: on the pool) on a group of G lanes (gl = the
// lane's place in it): a chunk of class c < LV_BIG holds 32 >> c variables,
// each on 2 << c lanes.  The variables of class LV_BIG come first, a
// workgroup to each.  A class is chosen from a bound on the words the
// variable needs; the staging checks the slice and falls back to the pool
// (one lane per variable).
template <class F>
__device__ inline void lv_chunks(const u32* work, u32* lds, F f) {
  const u32 lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const u32* placed = work + LV_WORK_HDR;
  u32 start[LV_CLASSES + 1];  // absent keys start where the next key starts
#pragma unroll
  for (u32 key = 0; key <= LV_CLASSES; key++) start[key] = work[key];
  constexpr u32 BIG = LV_CLASSES - 1 - LV_BIG;  // its key
  const u32 nbig = start[BIG + 1] - start[BIG];
  u32 chunks = 0;
#pragma unroll
  for (u32 key = 0; key < LV_CLASSES; key++) {
    const u32 L = lv_class_lanes(LV_CLASSES - 1 - key);
    if (key != BIG) chunks += (start[key + 1] - start[key] + L - 1) / L;
  }
  // the first chunks go to the workgroups after those of the large variables,
  // and to a workgroup's other wavefronts once every workgroup has one
  u32 J = (blockIdx.x + gridDim.x - nbig % gridDim.x) % gridDim.x + wave * gridDim.x;
  u32 big = wave ? nbig : blockIdx.x;
  bool shared = nbig != 0;  // the LDS is the first wavefront's until it is through with them
  while (true) {
    u32 r, s1, L, G, slice;
    u32* w = lds;
    if (big < nbig) {
      r = start[BIG] + big, s1 = r + 1, L = 1, G = 64, slice = LV_WAVES * LV_CAP;
      big += gridDim.x;
    } else {
      if (shared) __syncthreads();
      shared = false;
      if (J >= chunks) break;
      // the key of chunk J and its range, found by a loop over constant
      // indices so that start[] stays in registers (a loop that stops at the
      // key indexes it at run time, which puts the array in scratch memory)
      u32 key = LV_CLASSES - 1, j = J, s0 = start[LV_CLASSES - 1];
      s1 = start[LV_CLASSES];
      bool found = false;
#pragma unroll
      for (u32 q = 0; q < LV_CLASSES - 1; q++) {
        if (q == BIG) continue;
        const u32 Lq = lv_class_lanes(LV_CLASSES - 1 - q), m = (start[q + 1] - start[q] + Lq - 1) / Lq;
        if (!found) {
          if (j < m) {
            key = q, s0 = start[q], s1 = start[q + 1];
            found = true;
          } else {
            j -= m;
          }
        }
      }
      L = lv_class_lanes(LV_CLASSES - 1 - key), G = 64 / L, slice = LV_CAP / L;
      r = s0 + j * L + lane / G;
      w = key ? lds + wave * LV_CAP + lane / G * slice : nullptr;
      J += gridDim.x * LV_WAVES;
    }
    if (r < s1) f(placed[r], w, slice, lane % G, G);
    group_sync();  // the next chunk reuses the LDS
  }
}
// as many workgroups as the LDS lets onto the CUs, at most one per variable
constexpr u32 LV_BLOCKS = 256 * (160 * 1024 / LV_LDS);
// The least class of a launch over n variables: where they would leave
// lanes idle, each takes the largest group that keeps the launch within the
// lanes of LV_BLOCKS workgroups.  A variable's chain of dependent loads and
// LDS reads is then walked G entries at a time, and the chunks spread over
// the CUs.  Against a lane per variable, per launch (ve_decide_k, sub_k): 45
// elected variables 290 + 155 -> 48 + 27 us; 3,206: 350 + 260 -> 55 + 60 us.
// Twice and four times the lanes: 0.35 + 0.22 instead of 0.24 + 0.16 ms on
// 77,777 variables (three launches), 0.17 and 0.19 instead of 0.16 ms on
// 300,000, 0.59 and 0.55 instead of 0.60 ms on 100,000 gates (five).
static u32 lv_floor(u32 n) {
  u32 c = 0;
  while (c < LV_BIG - 1 && ((u64)n << (c + 2)) <= (u64)LV_BLOCKS * LV_WAVES * 64) c++;
  return c;
}

// VE decisions in one launch over every elected variable's staged lists: the
// gate checks (pure, equivalence, AND/OR), the ITE and XOR searches and the
// resolvent count.
// lsum[2k], lsum[2k + 1]: bounds on the clause size sums of the lists of
// elected variable k (from the list sort).  The searches' work grows with
// the square of the list lengths, their memory linearly: a variable's
// class is raised by VE_CLASS_BUMP (more lanes, a larger slice) over the
// class its lists need.
#ifndef VE_CLASS_BUMP
#define VE_CLASS_BUMP 1
#endif
struct VeClass {
  DB db;
  const u32 *pv, *lsum;
  u32 least, fine;
  __device__ u32 val(u32 k) const { return k; }
  __device__ u32 key(u32 k) const {
    const u32 p = V2L(pv[k]), w = db.ot_size[p] + db.ot_size[p | 1];
    const u64 b = lview_bound(w, (u64)lsum[2 * k] + lsum[2 * k + 1]);
    u32 c = lv_class(b);
    if (c < LV_BIG) c = max(least, min(c + VE_CLASS_BUMP, LV_BIG - 1));
    return ((LV_CLASSES - 1 - c) << LV_FINE_BITS) | (fine ? lv_fine(w) : 0u);
  }
};
// every elected variable on an LDS copy of its lists (the checks read each
// clause of the lists once, into LDS, instead of once per check from the
// pool), the gate checks, searches and resolvent count shared by the group
// (a few lanes or all 64 per variable).  Bound by chains of LDS
// reads per variable, so what counts is how many of them one lane walks.
__global__ void __launch_bounds__(LV_WAVES * 64) ve_decide_k(DB db, Options o, const u32* pv, VeDecision d,
                                                             const u32* work) {
  extern __shared__ u32 lds[];
  lv_chunks(work, lds, [&](u32 k, u32* w, u32 slice, u32 gl, u32 G) {
    const u32 v = pv[k];
    LView lv;
    if (w && lview_stage(db, v, w, slice, lv, gl, G)) {
      group_sync();
      ve_decide(lv, o, v, k, d, gl, G);
      group_sync();
      lview_commit(db, lv, gl, G);
    } else if (gl == 0) {
      ve_decide(db, o, v, k, d);
    }
  });
}
void k_ve_decide(const DB& db, const Options& o, const u32* pv, u32 n, const VeDecision& d, u32* work,
                 const u32* lsum, void* tmp, Stream* st) {
  if (!n) return;
  place(VeClass{db, pv, lsum, lv_floor(n), (u32)o.work_order}, n, 8, work + LV_WORK_HDR, work, LV_CLASSES + 1,
        LV_FINE_BITS, nullptr, 0, tmp, st);
  KLAUNCH_LDS(ve_decide_k, std::min<u32>(n, LV_BLOCKS), LV_WAVES * 64, LV_LDS, st, db, o, pv, d, work);
}
// SUB, staged as the VE searches (the class of a variable from the words of
// its SView, raised by SUB_CLASS_BUMP)
#ifndef SUB_CLASS_BUMP
#define SUB_CLASS_BUMP 0
#endif
struct SubClass {
  DB db;
  const u32 *pv, *idx, *lsum;
  u32 least, fine;
  __device__ u32 val(u32 t) const { return idx ? idx[t] : t; }
  __device__ u32 key(u32 t) const {
    const u32 k = val(t), p = V2L(pv[k]), w = db.ot_size[p] + db.ot_size[p | 1];
    const u64 b = sview_bound(w, (u64)lsum[2 * k] + lsum[2 * k + 1]);
    u32 c = lv_class(b);
    if (c < LV_BIG) c = max(least, min(c + SUB_CLASS_BUMP, LV_BIG - 1));
    return ((LV_CLASSES - 1 - c) << LV_FINE_BITS) | (fine ? lv_fine(w) : 0u);
  }
};
// take_snap: record each variable's state for the SUB re-runs just before
// its run (a run changes only the variable's own lists and clauses, so this
// equals a snapshot before the launch); the staged copy provides it
__global__ void __launch_bounds__(LV_WAVES * 64) sub_k(DB db, Options o, const u32* pv, const u32* work, SubOut out,
                                                       SubSnap snap, u32 take_snap) {
  extern __shared__ u32 lds[];
  lv_chunks(work, lds, [&](u32 k, u32* w, u32 slice, u32 gl, u32 G) {
    const u32 v = pv[k];
    SView sv;
    if (w && sview_stage(db, v, w, slice, sv, gl, G)) {
      group_sync();
      const u32 np0 = sv.w[0], nn0 = sv.w[1];
      if (take_snap) sub_snapshot_var(sv, v, k, snap, gl, G);
      group_sync();
      sub_var(sv, o, v, k, out, gl, G);
      group_sync();
      sview_commit(db, sv, np0, nn0, gl, G);
    } else if (gl == 0) {
      if (take_snap) sub_snapshot_var(db, v, k, snap);
      sub_var(db, o, v, k, out);
    }
  });
}
void k_sub(const DB& db, const Options& o, const u32* pv, const u32* idx, u32 n, const SubOut& out, u32* work,
           const u32* lsum, void* tmp, const SubSnap* snap, Stream* st) {
  if (!n) return;
  place(SubClass{db, pv, idx, lsum, lv_floor(n), (u32)o.work_order}, n, 8, work + LV_WORK_HDR, work,
        LV_CLASSES + 1, LV_FINE_BITS, out.n, 1, tmp, st);
  KLAUNCH_LDS(sub_k, std::min<u32>(n, LV_BLOCKS), LV_WAVES * 64, LV_LDS, st, db, o, pv, work, out,
              snap ? *snap : SubSnap{}, snap ? 1u : 0u);
}
// VE execution, staged as the searches: the resolvent path reads the
// variable's lists from LDS; EQU substitutions (which rewrite their clauses
// in place) work on the pool, EQU_CLASS lanes' worth or more each; variables
// VE keeps are not placed
constexpr u32 EQU_CLASS = 2;
struct ApplyClass {
  DB db;
  const u32 *pv, *type, *lsum;
  u32 least;
  __device__ u32 val(u32 t) const { return t; }
  __device__ u32 key(u32 k) const {
    if (!type[k]) return LV_CLASSES;
    u32 c = EQU_CLASS;
    if (type[k] != VT_EQU) {
      const u32 p = V2L(pv[k]);
      const u64 b = lview_bound(db.ot_size[p] + db.ot_size[p | 1], (u64)lsum[2 * k] + lsum[2 * k + 1]);
      c = lv_class(b);
    }
    if (c < LV_BIG) c = max(c, least);
    return LV_CLASSES - 1 - c;
  }
};
__global__ void __launch_bounds__(LV_WAVES * 64) ve_apply_k(DB db, const u32* pv, VeDecision d, VeApply a,
                                                            const u32* work) {
  extern __shared__ u32 lds[];
  lv_chunks(work, lds, [&](u32 k, u32* w, u32 slice, u32 gl, u32 G) {
    const u32 v = pv[k];
    LView lv;
    if (w && d.type[k] != VT_EQU && lview_stage(db, v, w, slice, lv, gl, G)) {
      group_sync();
      ve_apply(lv, db, v, k, d, a, gl, G);
    } else {
      ve_apply(db, db, v, k, d, a, gl, G);
    }
  });
}
void k_ve_apply(const DB& db, const u32* pv, u32 n, const VeDecision& d, const VeApply& a, u32* work,
                const u32* lsum, u32* zero, u32 nz, void* tmp, Stream* st) {
  if (!n) return;
  place(ApplyClass{db, pv, d.type, lsum, lv_floor(n)}, n, LV_KEY_BITS, work + LV_WORK_HDR, work, LV_CLASSES + 1,
        0, zero, nz, tmp, st);
  KLAUNCH_LDS(ve_apply_k, std::min<u32>(n, LV_BLOCKS), LV_WAVES * 64, LV_LDS, st, db, pv, d, a, work);
}
// in elected order (by score, so of similar lists): heaviest lists first took
// 0.69 instead of 0.61 ms for the two launches on 2.5M heavy-tailed variables
__global__ void bce_k(DB db, Options o, const u32* pv, const u32* type, u32 n, u32* words,
                      const u32* base, u32* stack, bool count) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  if (type && type[k]) {
    if (count) words[k] = 0;
    return;
  }
  if (count) words[k] = bce_var(db, o, pv[k], true, nullptr);
  else bce_var(db, o, pv[k], false, stack + base[k]);
}
void k_bce(const DB& db, const Options& o, const u32* pv, const u32* type, u32 n, u32* words,
           const u32* base, u32* stack, bool count, Stream* st) {
  if (!n) return;
  KLAUNCH(bce_k, grid_for(n, VB), VB, st, db, o, pv, type, n, words, base, stack, count);
}
__global__ void ere_k(DB db, Options o, const u32* pv, u32 from, u32 n, EreOut out) {
  const u32 k = from + blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) ere_var(db, o, pv[k], k, out);
}
void k_ere(const DB& db, const Options& o, const u32* pv, u32 from, u32 n, const EreOut& out, Stream* st) {
  if (from >= n) return;
  KLAUNCH(ere_k, grid_for(n - from, VB), VB, st, db, o, pv, from, n, out);
}
__global__ void ere_dirty_k(DB db, const u32* pv, u32 from, u32 n, const u32* del_by, u32* first) {
  const u32 k = from + blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n && ere_dirty_var(db, pv[k], k, del_by)) atomicMin(first, k);
}
void k_ere_dirty(const DB& db, const u32* pv, u32 from, u32 n, const u32* del_by, u32* first,
                 Stream* st) {
  if (from >= n) return;
  KLAUNCH(ere_dirty_k, grid_for(n - from, VB), VB, st, db, pv, from, n, del_by, first);
}
__global__ void del_by_k(const u32* rec, u32 nrec, u32* del_by) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nrec) atomicMin(&del_by[rec[3 * (u64)i + 2]], rec[3 * (u64)i]);
}
void k_del_by(const u32* rec, u32 nrec, u32* del_by, Stream* st) {
  if (!nrec) return;
  KLAUNCH(del_by_k, grid_for(nrec, 256), 256, st, rec, nrec, del_by);
}
__global__ void apply_del_k(DB db, const u32* ids, u32 n) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) set_deleted(db, ids[i]);
}
void k_apply_deletions(const DB& db, const u32* ids, u32 n, Stream* st) {
  if (!n) return;
  KLAUNCH(apply_del_k, grid_for(n, 256), 256, st, db, ids, n);
}
__global__ void ht_build_k(DB db, HashTable ht, int maxsize) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls) ht_insert_clause(db, ht, db.c_off[i], maxsize);
}
void k_ht_build(const DB& db, const HashTable& ht, int maxsize, Stream* st) {
  fill_u32((u32*)ht.slot, 0xFFFFFFFFu, 2 * ((size_t)ht.mask + 1), st);
  if (!db.ncls) return;
  KLAUNCH(ht_build_k, grid_for(db.ncls, 256), 256, st, db, ht, maxsize);
}
__global__ void ere_pair_counts_k(DB db, Options o, const u32* pv, u32 n, u32* np, unsigned long long* total) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long c = 0;
  if (k < n) {
    c = ere_pair_count(db, o, pv[k]);
    np[k] = (u32)c;
  }
  c = wave_sum64(c);
  if ((threadIdx.x & 63) == 0 && c) atomicAdd(total, c);
}
void k_ere_pair_counts(const DB& db, const Options& o, const u32* pv, u32 n, u32* np, u64* total, Stream* st) {
  fill_u32((u32*)total, 0, 2, st);
  if (!n) return;
  KLAUNCH(ere_pair_counts_k, grid_for(n, 256), 256, st, db, o, pv, n, np, (unsigned long long*)total);
}
// one thread per resolvent pair; the owning variable is found by a binary
// search over the per-variable pair offsets
__global__ void ere_pairs_k(DB db, ErePairs a, u32 npairs) {
  const u32 t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= npairs) return;
  u32 lo = 0, hi = a.nvars;  // first k with pbase[k] > t
  while (lo < hi) {
    const u32 mid = (lo + hi) >> 1;
    if (a.pbase[mid] <= t) lo = mid + 1;
    else hi = mid;
  }
  const u32 k = lo - 1;
  ere_pair(db, a, k, t - a.pbase[k]);
}
void k_ere_pairs(const DB& db, const ErePairs& a, u32 npairs, Stream* st) {
  if (!npairs) return;
  KLAUNCH(ere_pairs_k, grid_for(npairs, 256), 256, st, db, a, npairs);
}
__global__ void ere_all_matches_k(DB db, ErePairs a, u32 n, const u32* off, u32* out) {
  const u32 o = blockIdx.x * blockDim.x + threadIdx.x;
  if (o < n) ere_all_matches(db, a, o, off, out);
}
void k_ere_all_matches(const DB& db, const ErePairs& a, u32 n, const u32* off, u32* out, Stream* st) {
  if (!n) return;
  KLAUNCH(ere_all_matches_k, grid_for(n, 64), 64, st, db, a, n, off, out);
}

// ---------------------------------------------------------------- small helpers
__global__ void assign_units_k(DB db, const u32* lits, u32 n) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const u32 l = lits[i];
  db.assign[ABS(l)] = l + 1;
  db.vstate[ABS(l)] = VS_FROZEN;
}
void k_assign_units(const DB& db, const u32* lits, u32 n, Stream* st) {
  if (!n) return;
  KLAUNCH(assign_units_k, grid_for(n, 256), 256, st, db, lits, n);
}
__global__ void max_list_k(DB db, const u32* lits, u32 n, u32* out) {
  u32 m = 0;
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    m = max(m, db.ot_size[lits[i]]);
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) atomicMax(out, m);
}
void k_max_list(const DB& db, const u32* lits, u32 n, u32* out, Stream* st) {
  fill_u32(out, 0, 1, st);
  if (!n) return;
  KLAUNCH(max_list_k, std::min(grid_for(n, 256), RED_BLOCKS), 256, st, db, lits, n, out);
}
__global__ void reduce_lists_k(DB db) {
  const u32 l = blockIdx.x * blockDim.x + threadIdx.x + 2;
  if (l >= 2 * db.nvars + 2) return;
  u32* r = db.ot_refs + db.ot_off[l];
  const u32 n = db.ot_size[l];
  u32 j = 0;
  for (u32 i = 0; i < n; i++)
    if (!is_deleted(db, r[i])) r[j++] = r[i];
  db.ot_size[l] = j;
}
void k_reduce_lists(const DB& db, Stream* st) {
  KLAUNCH(reduce_lists_k, grid_for(2 * (size_t)db.nvars, 256), 256, st, db);
}
// literals sorted, signature
__device__ inline void prep_clause(u32* h, u32 n) {
  u32* l = h + CL_HDR;
  for (u32 q = 1; q < n; q++) {
    const u32 t = l[q];
    u32 j = q;
    while (j > 0 && l[j - 1] > t) { l[j] = l[j - 1]; j--; }
    l[j] = t;
  }
  h[1] = calc_sig(l, n);
}
__global__ void prep_k(DB db, u32 first) {
  const u32 i = first + blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= db.ncls) return;
  u32* h = chead(db, db.c_off[i]);
  prep_clause(h, hdr_size(h[0]));
}
__global__ void raw_learnt_k(RawClauses r) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= r.n) return;
  const bool learnt = r.flags[i] & 1;
  r.lrank[i] = learnt ? 1u : 0u;
  r.lwords[i] = learnt ? CL_HDR + (u32)(r.off[i + 1] - r.off[i]) : 0u;
}
// a thread per clause: its place is what precedes it in the given order, less
// the learnt clauses among that, or for a learnt clause all originals and the
// learnt ones before it
__global__ void raw_build_k(DB db, RawClauses r) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= r.n) return;
  const u64 o0 = r.off[i] - r.off[0];
  const u32 n = (u32)(r.off[i + 1] - r.off[i]);
  const u8 f = r.flags ? r.flags[i] : 0;
  const bool learnt = f & 1;
  u32 at = i, handle = CL_HDR * i + (u32)o0;
  if (r.flags) {
    const u32 lr = r.lrank[i], lw = r.lwords[i];
    at = learnt ? r.n - r.sc[1] + lr : at - lr;
    handle = learnt ? r.words - r.sc[2] + lw : handle - lw;
  }
  u32* h = db.lits + handle;
  const u32* src = r.lits + o0;
  db.c_off[at] = handle;
  h[0] = make_hdr(n, learnt ? (u8)(ST_LEARNT | (f & USAGE_MASK)) : (u8)ST_ORIGINAL);
  h[2] = learnt && r.lbd ? (r.lbd[i] & 0x03FFFFFFu) : 0u;
  bool bad = false;
  for (u32 q = 0; q < n; q++) {
    const u32 l = src[q];
    bad |= ABS(l) == 0 || ABS(l) > r.maxvar;
    u32 j = q;  // insertion into the sorted literals before it
    while (j > 0 && h[CL_HDR + j - 1] > l) {
      h[CL_HDR + j] = h[CL_HDR + j - 1];
      j--;
    }
    h[CL_HDR + j] = l;
  }
  h[1] = calc_sig(h + CL_HDR, n);
  if (bad) *r.sc = 1;
}
void k_build_clauses(const DB& db, const RawClauses& raw, void* tmp, Stream* st) {
  if (!raw.n) return;
  if (raw.flags) {
    KLAUNCH(raw_learnt_k, grid_for(raw.n, 256), 256, st, raw);
    scan_set(ScanSet{{raw.lrank, raw.lwords}, {raw.lrank, raw.lwords}, {raw.sc + 1, raw.sc + 2}}, 2, raw.n, tmp, st);
  }
  KLAUNCH(raw_build_k, grid_for(raw.n, 256), 256, st, db, raw);
}
// Appended clauses.  A host loop takes 9.4 ns per clause (0.62 ms for the
// 66,000 clauses of ten frames, 0.178 here with the copies); a thread per
// clause, with the order of the units settled by repeated passes:
// a clause sees the units of earlier clauses as the pass before found them, so
// pass p is right for every chain of p units, and nothing changes any more
// once it is right for all (7 passes of 3-4 us for those frames).  Clauses
// longer than AP_LONG (quadratic in one thread) are left to the host.
__global__ void append_pass_k(DB db, AppendArgs a, u32 pass) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n || !append_runs(a, pass)) return;
  const u64 any = __ballot(append_pass(db, a, i, pass));
  if (any && (threadIdx.x & 63) == (u32)__builtin_ctzll(any)) a.fl[AP_CHANGED + pass] = 1;
}
__global__ void append_write_k(DB db, AppendArgs a, u32 last, u32 c0, u32 w0) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < a.n) append_write(db, a, i, last, c0, w0);
}
void k_append_pass(const DB& db, const AppendArgs& a, u32 pass, Stream* st) {
  KLAUNCH(append_pass_k, grid_for(a.n, 256), 256, st, db, a, pass);
}
void k_append_place(const AppendArgs& a, void* tmp, Stream* st) {
  scan_set(ScanSet{{a.kept, a.words}, {a.kept, a.words}, {a.fl + 4, a.fl + 5}}, 2, a.n, tmp, st);
}
void k_append_write(const DB& db, const AppendArgs& a, u32 last, u32 c0, u32 w0, Stream* st) {
  KLAUNCH(append_write_k, grid_for(a.n, 256), 256, st, db, a, last, c0, w0);
}
void k_prep(const DB& db, u32 first, Stream* st) {
  if (first >= db.ncls) return;
  KLAUNCH(prep_k, grid_for(db.ncls - first, 256), 256, st, db, first);
}
__global__ void clear_added_k(DB db) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= db.ncls) return;
  const u32 c = db.c_off[i];
  const u8 f = cflags(db, c);
  if (f & F_ADDED) set_cflags(db, c, (u8)(f & ~F_ADDED));
}
void k_clear_added(const DB& db, Stream* st) {
  if (!db.ncls) return;
  KLAUNCH(clear_added_k, grid_for(db.ncls, 256), 256, st, db);
}
__global__ void zero_sizes_k(DB db, const u32* lits, u32 n) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) db.ot_size[lits[i]] = 0;
}
void k_zero_sizes(const DB& db, const u32* lits, u32 n, Stream* st) {
  if (!n) return;
  KLAUNCH(zero_sizes_k, grid_for(n, 256), 256, st, db, lits, n);
}

// ---------------------------------------------------------------- DRAT proof
__global__ void proof_sizes_k(DB db, const u32* lines, u32 n, const u32* stamp, u32* bytes) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) bytes[i] = proof_line_size(db, lines, i, stamp);
}
__global__ void proof_write_k(DB db, const u32* lines, u32 n, const u32* bytes, const u32* off, u8* out) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && bytes[i]) proof_line_write(db, lines, i, out + off[i]);  // 0 bytes: dropped line
}
void k_proof_sizes(const DB& db, const u32* lines, u32 n, const u32* stamp, u32* bytes, Stream* st) {
  if (!n) return;
  KLAUNCH(proof_sizes_k, grid_for(n, 256), 256, st, db, lines, n, stamp, bytes);
}
void k_proof_write(const DB& db, const u32* lines, u32 n, const u32* bytes, const u32* off, u8* out,
                   Stream* st) {
  if (!n) return;
  KLAUNCH(proof_write_k, grid_for(n, 256), 256, st, db, lines, n, bytes, off, out);
}
__global__ void set_stamps_k(u32* stamp, const u32* pairs, u32 n, int clear) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) stamp[pairs[2 * i]] = clear ? 0u : pairs[2 * i + 1];
}
void k_set_stamps(u32* stamp, const u32* pairs, u32 n, bool clear, Stream* st) {
  if (!n) return;
  KLAUNCH(set_stamps_k, grid_for(n, 256), 256, st, stamp, pairs, n, clear ? 1 : 0);
}

// ---------------------------------------------------------------- count / compact
// adds the workgroup's values to *out with one atomic: one per wavefront of
// 1,024 workgroups, 8,192 on the two words, were most of the 70 us that
// counting 160,000 clauses took
__device__ inline void block_add64(unsigned long long x, unsigned long long* out) {
  __shared__ unsigned long long lw[ST / 64];
  x = wave_sum64(x);
  if ((threadIdx.x & 63) == 0) lw[threadIdx.x >> 6] = x;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (u32 w = 1; w < ST / 64; w++) x += lw[w];
    if (x) atomicAdd(out, x);
  }
  __syncthreads();
}
__global__ void __launch_bounds__(ST) count_k(DB db, unsigned long long* out) {
  unsigned long long live = 0, lits = 0;
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < db.ncls; i += gridDim.x * blockDim.x) {
    const u32 h = chead(db, db.c_off[i])[0];
    if (!st_deleted(hdr_flags(h))) {
      live++;
      lits += hdr_size(h);
    }
  }
  block_add64(live, &out[0]);
  block_add64(lits, &out[1]);
}
// occurrences (O_E) and clause bytes (D_E: 12-byte header + 4 bytes per
// literal) of the live clauses in the elected variables' lists; elected
// variables share no clause, so every clause is counted once
__global__ void elected_work_k(DB db, const u32* pv, u32 n, unsigned long long* out) {
  unsigned long long occ = 0, bytes = 0;
  for (u32 k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    for (u32 s = 0; s < 2; s++) {
      const OLV ol = olist(db, V2L(pv[k]) | s);
      for (u32 i = 0; i < ol.n; i++) {
        const u32 h = chead(db, ol.r[i])[0];
        if (st_deleted(hdr_flags(h))) continue;
        occ++;
        bytes += 12 + 4ull * hdr_size(h);
      }
    }
  }
  occ = wave_sum64(occ);
  bytes = wave_sum64(bytes);
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&out[0], occ);
    atomicAdd(&out[1], bytes);
  }
}
// occurrences in the election candidates' lists (O_c) with their clauses
// marked (per handle), then the bytes of the distinct marked clauses (D_c);
// the marks are cleared again.  Profiling only.
__global__ void cand_occ_k(DB db, const u32* cand, u32 n, u8* mark, unsigned long long* out) {
  unsigned long long occ = 0;
  for (u32 k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
    for (u32 s = 0; s < 2; s++) {
      const OLV ol = olist(db, V2L(cand[k]) | s);
      for (u32 i = 0; i < ol.n; i++) {
        const u32 c = ol.r[i];
        if (st_deleted(hdr_flags(chead(db, c)[0]))) continue;
        occ++;
        mark[c] = 1;
      }
    }
  }
  occ = wave_sum64(occ);
  if ((threadIdx.x & 63) == 0) atomicAdd(&out[0], occ);
}
__global__ void marked_bytes_k(DB db, u8* mark, unsigned long long* out) {
  unsigned long long bytes = 0;
  for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < db.ncls; i += gridDim.x * blockDim.x) {
    const u32 c = db.c_off[i];
    if (!mark[c]) continue;
    mark[c] = 0;
    bytes += 12 + 4ull * csize(db, c);
  }
  bytes = wave_sum64(bytes);
  if ((threadIdx.x & 63) == 0) atomicAdd(&out[1], bytes);
}
void k_cand_work(const DB& db, const u32* cand, u32 n, u8* mark, u64* out2, Stream* st) {
  fill_u32((u32*)out2, 0, 4, st);
  if (!n) return;
  KLAUNCH(cand_occ_k, std::min(grid_for(n, ST), RED_BLOCKS), ST, st, db, cand, n, mark, (unsigned long long*)out2);
  if (db.ncls)
    KLAUNCH(marked_bytes_k, std::min(grid_for(db.ncls, ST), RED_BLOCKS), ST, st, db, mark,
            (unsigned long long*)out2);
}
void k_elected_work(const DB& db, const u32* pv, u32 n, u64* out2, Stream* st) {
  fill_u32((u32*)out2, 0, 4, st);
  if (!n) return;
  KLAUNCH(elected_work_k, std::min(grid_for(n, ST), RED_BLOCKS), ST, st, db, pv, n, (unsigned long long*)out2);
}
void k_count(const DB& db, u64* out2, Stream* st) {
  fill_u32((u32*)out2, 0, 4, st);
  if (!db.ncls) return;
  KLAUNCH(count_k, std::min(grid_for(db.ncls, 4 * ST), RED_BLOCKS), ST, st, db, (unsigned long long*)out2);
}
// sel: 0 every live clause, 1 live originals only, 2 live learnt clauses only
__device__ inline bool compact_sel(u32 h, int sel) {
  const u8 f = hdr_flags(h);
  if (st_deleted(f)) return false;
  return sel == 0 || (sel == 1) == !st_learnt(f);
}
__global__ void live_k(DB db, u32* tc, u32* tl, int sel) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= db.ncls) return;
  const u32 h = chead(db, db.c_off[i])[0];
  const bool live = compact_sel(h, sel);
  tc[i] = live ? 1u : 0u;
  tl[i] = live ? CL_HDR + hdr_size(h) : 0u;  // pool words
}
// base (device, nullable): clause index and pool word where the selection starts
__global__ void compact_k(DB src, DB dst, const u32* tc, const u32* tl, int sel, const u32* base) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= src.ncls) return;
  const u32* a = chead(src, src.c_off[i]);
  const u32 h = a[0];
  if (!compact_sel(h, sel)) return;
  const u32 nid = tc[i] + (base ? base[0] : 0u), noff = tl[i] + (base ? base[1] : 0u), n = hdr_size(h);
  dst.c_off[nid] = noff;
  u32* b = dst.lits + noff;
  b[0] = make_hdr(n, (u8)(hdr_flags(h) & ~F_MOLTEN));
  for (u32 i = 1; i < CL_HDR + n; i++) b[i] = a[i];
}
void k_compact(const DB& src, DB& dst, u32* tmp_cls, u32* tmp_lit, void* tmp, u32* totals, Stream* st) {
  if (!src.ncls) {
    fill_u32(totals, 0, 2, st);
    return;
  }
  KLAUNCH(live_k, grid_for(src.ncls, 256), 256, st, src, tmp_cls, tmp_lit, 0);
  scan_u32(tmp_cls, tmp_cls, src.ncls, totals, tmp, st);
  scan_u32(tmp_lit, tmp_lit, src.ncls, totals + 1, tmp, st);
  KLAUNCH(compact_k, grid_for(src.ncls, 256), 256, st, src, dst, tmp_cls, tmp_lit, 0, (const u32*)nullptr);
}
// the live clauses with the originals first and the learnt clauses after
// them, each part in clause order (totals[0..1]: clauses and words in all;
// totals[2..3] scratch)
__global__ void add_totals_k(u32* t) {
  t[0] += t[2];
  t[1] += t[3];
}
void k_compact_originals_first(const DB& src, DB& dst, u32* tmp_cls, u32* tmp_lit, void* tmp, u32* totals,
                               Stream* st) {
  if (!src.ncls) {
    fill_u32(totals, 0, 4, st);
    return;
  }
  KLAUNCH(live_k, grid_for(src.ncls, 256), 256, st, src, tmp_cls, tmp_lit, 1);
  scan_u32(tmp_cls, tmp_cls, src.ncls, totals, tmp, st);
  scan_u32(tmp_lit, tmp_lit, src.ncls, totals + 1, tmp, st);
  KLAUNCH(compact_k, grid_for(src.ncls, 256), 256, st, src, dst, tmp_cls, tmp_lit, 1, (const u32*)nullptr);
  KLAUNCH(live_k, grid_for(src.ncls, 256), 256, st, src, tmp_cls, tmp_lit, 2);
  scan_u32(tmp_cls, tmp_cls, src.ncls, totals + 2, tmp, st);
  scan_u32(tmp_lit, tmp_lit, src.ncls, totals + 3, tmp, st);
  KLAUNCH(compact_k, grid_for(src.ncls, 256), 256, st, src, dst, tmp_cls, tmp_lit, 2, (const u32*)totals);
  KLAUNCH(add_totals_k, 1, 1, st, totals);
}

// ---------------------------------------------------------------- variable map
// First root-assigned variable (VMAP::initiate, src/cpu/vmap.h:63-77): the
// lowest set lane of a wave holds the wave's smallest candidate, so each
// wave issues at most one atomic.
__global__ void map_first_k(const u8* vstate, const u32* assign, u32 nvars, u32* first) {
  const u32 v = blockIdx.x * blockDim.x + threadIdx.x + 1;
  const bool cand = v <= nvars && vstate[v] && assign[v];
  const unsigned long long b = __ballot(cand);
  // a wave whose smallest candidate cannot win skips the atomic
  if (cand && (u32)(__ffsll(b) - 1) == (threadIdx.x & 63u) && v < __atomic_load_n(first, __ATOMIC_RELAXED))
    atomicMin(first, v);
}
__global__ void map_keep_k(const u8* vstate, u32 nvars, const u32* first, u32* keep) {
  const u32 v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v > nvars) return;
  const u32 f = *first == 0xFFFFFFFFu ? 0u : *first;
  keep[v] = map_keep(vstate, v, f);
}
// pos: exclusive scan of the keep flags -> mapped
__global__ void map_index_k(const u8* vstate, u32 nvars, const u32* first, const u32* pos, u32* mapped) {
  const u32 v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v > nvars) return;
  const u32 f = *first == 0xFFFFFFFFu ? 0u : *first;
  mapped[v] = map_keep(vstate, v, f) ? pos[v] + 1 : 0u;
}
// info = {first (0: none), new variable count, true literal of first, inactive variables}
__global__ void map_info_k(const u32* assign, const u32* mapped, u32 nvars, const u32* total, u32* info) {
  const u32 f = info[0] == 0xFFFFFFFFu ? 0u : info[0];
  const u32 n = *total;
  info[0] = f;
  info[1] = n;
  info[2] = f ? (V2L(mapped[f]) | SIGN(assign[f] - 1)) : 0u;
  info[3] = nvars - (n - (f ? 1u : 0u));
}
void k_map_build(const u8* vstate, const u32* assign, u32 nvars, u32* pos_tmp, u32* mapped, u32* info,
                 void* tmp, Stream* st) {
  fill_u32(info, 0xFFFFFFFFu, 1, st);
  if (nvars) KLAUNCH(map_first_k, grid_for(nvars, 256), 256, st, vstate, assign, nvars, info);
  KLAUNCH(map_keep_k, grid_for((size_t)nvars + 1, 256), 256, st, vstate, nvars, info, pos_tmp);
  scan_u32(pos_tmp, pos_tmp, (size_t)nvars + 1, info + 4, tmp, st);
  KLAUNCH(map_index_k, grid_for((size_t)nvars + 1, 256), 256, st, vstate, nvars, info, pos_tmp, mapped);
  KLAUNCH(map_info_k, 1, 1, st, assign, mapped, nvars, info + 4, info);
}
__global__ void map_clauses_k(DB db, VarMap m) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls) map_clause(db, db.c_off[i], m);
}
void k_map_clauses(const DB& db, const VarMap& m, Stream* st) {
  if (!db.ncls) return;
  KLAUNCH(map_clauses_k, grid_for(db.ncls, 256), 256, st, db, m);
}
// per-variable arrays in the new numbering (VMAP::mapShrinkVars and mapSP,
// vmap.h:80-100, 132-143): only 'first' stays assigned
__global__ void map_vars_k(VarMap m, u32 nvars_old, const u32* vorg, const u8* vstate, const u8* assumed,
                           u32* vorg2, u8* vstate2, u8* assumed2, u32* assign2) {
  const u32 v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v > nvars_old) return;
  if (v == 0) {
    vorg2[0] = vorg[0];
    vstate2[0] = 0;
    assumed2[0] = 0;
    assign2[0] = 0;
    return;
  }
  const u32 nv = m.mapped[v];
  if (!nv) return;
  vorg2[nv] = vorg[v];
  vstate2[nv] = vstate[v];
  assumed2[nv] = assumed[v];
  assign2[nv] = v == m.first ? m.first_true + 1 : 0u;
}
void k_map_vars(const VarMap& m, u32 nvars_old, const u32* vorg, const u8* vstate, const u8* assumed, u32* vorg2,
                u8* vstate2, u8* assumed2, u32* assign2, Stream* st) {
  KLAUNCH(map_vars_k, grid_for((size_t)nvars_old + 1, 256), 256, st, m, nvars_old, vorg, vstate, assumed, vorg2,
          vstate2, assumed2, assign2);
}
// VMAP::mapOrgs (vmap.h:112-131): 0 stays 0
__global__ void map_lits_k(VarMap m, u32* lits, u64 n) {
  const u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && lits[i]) lits[i] = map_lit(m, lits[i]);
}
void k_map_lits(const VarMap& m, u32* lits, u64 n, Stream* st) {
  if (!n) return;
  KLAUNCH(map_lits_k, grid_for(n, 256), 256, st, m, lits, n);
}

// ---------------------------------------------------------------- fixed device scratch
// Staging memory of the entry points that allocate nothing
// (pfs_map_lits_noalloc): one array per device, held until the process
// ends.  Host code never uses the array's name as an address: its device
// address is looked up once per device (hipGetSymbolAddress, with that
// device current) and kept.  Every call on a device shares the array, so
// calls that overlap on one device race.
static __device__ __align__(256) u32 scratch[SCRATCH_WORDS];
static std::mutex g_scratch_m;
static std::map<int, u32*> g_scratch;
u32* scratch_lookup(int device) {
  std::lock_guard<std::mutex> lk(g_scratch_m);
  auto it = g_scratch.find(device);
  if (it != g_scratch.end()) return it->second;
  int cur = -1;
  PFS_HIP(hipGetDevice(&cur));
  if (cur != device) throw std::runtime_error("scratch lookup: device " + std::to_string(device) + " is not current");
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    (void)hipGetLastError();
    throw std::runtime_error(std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
  }
  g_scratch[device] = (u32*)p;
  return (u32*)p;
}

// ---------------------------------------------------------------- output packing
__global__ void pack_sizes_k(DB db, u32* sizes) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls) sizes[i] = csize(db, db.c_off[i]);
}
__global__ void pack_k(DB db, const u32* start, u64* offsets, u32* lits, u8* flags, u32* lbd) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls) pack_clause(db, i, start, offsets, lits, flags, lbd);
}
void k_pack_cnf(const DB& db, u32* start_tmp, void* tmp, u32* total, u64* offsets, u32* lits, u8* flags, u32* lbd,
                Stream* st) {
  if (!db.ncls) {
    fill_u32((u32*)offsets, 0, 2, st);
    return;
  }
  KLAUNCH(pack_sizes_k, grid_for(db.ncls, 256), 256, st, db, start_tmp);
  scan_u32(start_tmp, start_tmp, db.ncls, total, tmp, st);
  KLAUNCH(pack_k, grid_for(db.ncls, 256), 256, st, db, start_tmp, offsets, lits, flags, lbd);
}

// ---------------------------------------------------------------- DIMACS ingestion
// The clause part of a DIMACS text (src/cpu/dimacs.cpp:41-110, toClause
// :113-170) is lexed on the device in 4096-byte tiles: workgroup b owns
// bytes [4096 b, 4096 b + 4096) of the text, each of its 256 threads 16
// consecutive bytes read with one 16-byte load (the text buffer is padded
// with blanks to whole tiles).  A token starts at a byte that is not blank
// (bytes 9-13 and 32, dimacs.h:33) and follows a blank or the start of the
// clause part.  Bytes of comment lines ('c' tokens, to the end of the line)
// are masked; the clause part ends at the first NUL byte or '%' token.
constexpr u32 LEX_T = 256, LEX_B = 16, LEX_TILE = LEX_T * LEX_B;
template <u32 MODE>
__global__ void __launch_bounds__(LEX_T) lex_k(LexArgs a) {
  __shared__ u32 lw[NW];
  const u64 base = (u64)blockIdx.x * LEX_TILE + (u64)threadIdx.x * LEX_B;
  const uint4 w = *(const uint4*)(a.text + base);
  u8 b[LEX_B];
  *(uint4*)b = w;
  u32 prev = base ? a.text[base - 1] : 32u;
  u32 mine = 0;  // starts of the kind this mode counts or emits
  u32 kinds = 0;  // bit j: byte j starts such a token
#pragma unroll
  for (u32 j = 0; j < LEX_B; j++) {
    const u64 i = base + j;
    const u32 c = b[j];
    const bool start = lex_start(i, c, prev, a.begin, a.end);
    prev = c;
    if (MODE == LEX_SPECIAL) {
      if (i >= a.begin && i < a.end && c == 0) atomicMin(&a.mark[0], (unsigned long long)i);
      if (start && c == '%') atomicMin(&a.mark[1], (unsigned long long)i);
      if (start && c == 'c') kinds |= 1u << j;
    } else if (MODE == LEX_COMMENTS) {
      if (start && c == 'c') kinds |= 1u << j;
    } else if (MODE == LEX_PERCENT) {
      if (start && c == '%' && !a.mask[i]) atomicMin(&a.mark[1], (unsigned long long)i);
    } else {
      if (start && c != 0 && !(a.mask && a.mask[i])) kinds |= 1u << j;
    }
  }
  mine = __popc(kinds);
  if (MODE == LEX_PERCENT) return;
  u32 tot;
  const u32 pre = block_excl_scan(mine, lw, &tot);
  if (MODE == LEX_SPECIAL || MODE == LEX_COUNT) {
    if (threadIdx.x == 0) a.cnt[blockIdx.x] = tot;
    return;
  }
  u32 k = a.cnt[blockIdx.x] + pre;
  while (kinds) {
    const u32 j = __ffs(kinds) - 1;
    kinds &= kinds - 1;
    const u64 i = base + j;
    if (MODE == LEX_COMMENTS) {
      a.pos[k++] = i;
      continue;
    }
    bool bad, big;
    a.lits[k++] = lex_literal(a.text, i, a.end, a.maxvar, bad, big);
    if (bad) {
      atomicOr(a.err, (u32)LEXE_TOKEN);
      atomicMin(&a.mark[2], (unsigned long long)i);
    }
    if (big) atomicOr(a.err, (u32)LEXE_VAR);  // "too many variables"
  }
}
// one thread per comment start: its bytes up to and including the newline
__global__ void lex_mask_k(const u8* text, u64 end, const u64* pos, u32 n, u8* mask) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  for (u64 i = pos[k]; i < end; i++) {
    mask[i] = 1;
    if (text[i] == '\n') break;
  }
}
u64 lex_tiles(u64 n) { return (n + LEX_TILE - 1) / LEX_TILE; }
void k_lex(u32 mode, const LexArgs& a, u64 ntiles, Stream* st) {
  if (!ntiles) return;
  switch (mode) {
    case LEX_SPECIAL: KLAUNCH(lex_k<LEX_SPECIAL>, (unsigned)ntiles, LEX_T, st, a); break;
    case LEX_COMMENTS: KLAUNCH(lex_k<LEX_COMMENTS>, (unsigned)ntiles, LEX_T, st, a); break;
    case LEX_PERCENT: KLAUNCH(lex_k<LEX_PERCENT>, (unsigned)ntiles, LEX_T, st, a); break;
    case LEX_COUNT: KLAUNCH(lex_k<LEX_COUNT>, (unsigned)ntiles, LEX_T, st, a); break;
    default: KLAUNCH(lex_k<LEX_EMIT>, (unsigned)ntiles, LEX_T, st, a); break;
  }
}
void k_lex_mask(const u8* text, u64 end, const u64* pos, u32 n, u8* mask, Stream* st) {
  if (!n) return;
  KLAUNCH(lex_mask_k, grid_for(n, 256), 256, st, text, end, pos, n, mask);
}
// clause ends: ends[c] = index of the c-th 0 among the literals
__global__ void zero_flags_k(const u32* lits, u64 n, u32* z) {
  const u64 k = (u64)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) z[k] = lits[k] == 0;
}
__global__ void zero_emit_k(const u32* lits, u64 n, const u32* pos, u32* ends) {
  const u64 k = (u64)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n && lits[k] == 0) ends[pos[k]] = (u32)k;
}
void k_clause_ends(const u32* lits, u64 n, u32* tmp_pos, void* tmp, u32* total, u32* ends, Stream* st) {
  if (!n) {
    fill_u32(total, 0, 1, st);
    return;
  }
  KLAUNCH(zero_flags_k, grid_for(n, 256), 256, st, lits, n, tmp_pos);
  scan_u32(tmp_pos, tmp_pos, n, total, tmp, st);
  KLAUNCH(zero_emit_k, grid_for(n, 256), 256, st, lits, n, tmp_pos, ends);
}
// clause i holds the literals between the (i-1)-th and the i-th 0; in the
// pool it starts at that literal offset plus two words per earlier clause
__global__ void parse_build_k(DB db, const u32* lits, const u32* ends, u32* err) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls && !parse_build_clause(db, lits, ends, i)) atomicOr(err, (u32)LEXE_SIZE);
}
void k_parse_build(const DB& db, const u32* lits, const u32* ends, u32* err, Stream* st) {
  if (!db.ncls) return;
  KLAUNCH(parse_build_k, grid_for(db.ncls, 256), 256, st, db, lits, ends, err);
}
// ingestion proof: bytes per line (units first, then the text clauses),
// then the lines at their scanned offsets
__global__ void parse_proof_k(DB db, const u32* toks, const u32* ends, const u32* units, u32 nu, u32 nc,
                              const u32* off, u8* out, u32* bytes) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nu + nc) return;
  u8* o = off ? out + off[i] : nullptr;
  const u32 b = i < nu ? unit_proof_line(db, units[i], o) : parse_proof_clause(db, toks, ends, i - nu, o);
  if (!off) bytes[i] = b;
}
void k_parse_proof(const DB& db, const u32* toks, const u32* ends, const u32* units, u32 nu, u32 nc,
                   const u32* off, u8* out, u32* bytes, Stream* st) {
  if (!(nu + nc)) return;
  KLAUNCH(parse_proof_k, grid_for((size_t)nu + nc, 256), 256, st, db, toks, ends, units, nu, nc, off, out, bytes);
}
// rewrite proof: line i < nu is unit i, then the additions (phase 0) of
// clause indices 0..ncls, then the deletions (phase 1)
__global__ void rewrite_proof_k(DB db, const u32* old, const u32* units, u32 nu, const u32* off, u8* out,
                                u32* bytes) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nu + 2 * db.ncls) return;
  u8* o = off ? out + off[i] : nullptr;
  u32 b;
  if (i < nu) {
    b = unit_proof_line(db, units[i], o);
  } else {
    const u32 j = i - nu, phase = j >= db.ncls;
    b = rewrite_proof_clause(db, old, db.c_off[phase ? j - db.ncls : j], (int)phase, o);
  }
  if (!off) bytes[i] = b;
}
void k_rewrite_proof(const DB& db, const u32* old, const u32* units, u32 nu, const u32* off, u8* out, u32* bytes,
                     Stream* st) {
  const size_t n = (size_t)nu + 2 * (size_t)db.ncls;
  if (!n) return;
  KLAUNCH(rewrite_proof_k, grid_for(n, 256), 256, st, db, old, units, nu, off, out, bytes);
}
// after the literal sort: duplicates dropped, tautologies removed, empty
// clauses reported, unit clauses turned into unit records (toClause,
// dimacs.cpp:120-166); ulit[i] = the unit literal of clause i or 0;
// kept[0] counts the clauses that stay
__global__ void parse_dedup_k(DB db, u32* ulit, u32* err) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls && parse_dedup_clause(db, db.c_off[i], &ulit[i]) == 2) atomicOr(err, (u32)LEXE_UNSAT);
}
void k_parse_dedup(const DB& db, u32* ulit, u32* err, Stream* st) {
  if (!db.ncls) return;
  KLAUNCH(parse_dedup_k, grid_for(db.ncls, 256), 256, st, db, ulit, err);
}
// unit clauses in text order: the first one of each variable is assigned
// (enqueueUnit); a later one of the other sign is a conflict
__global__ void parse_claim_k(const u32* ulit, u32 n, u32* first) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && ulit[i]) atomicMin(&first[ABS(ulit[i])], i);
}
__global__ void parse_settle_k(const u32* ulit, u32 n, const u32* first, u32* win, u32* err) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const u32 u = ulit[i];
  win[i] = 0;
  if (!u) return;
  const u32 f = first[ABS(u)];
  if (ulit[f] != u) atomicOr(err, (u32)LEXE_UNSAT);
  win[i] = f == i;
}
__global__ void parse_trail_k(DB db, const u32* ulit, u32 n, const u32* win, const u32* pos, u32* trail) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !win[i]) return;
  const u32 u = ulit[i];
  trail[pos[i]] = u;
  db.assign[ABS(u)] = u + 1;
  db.vstate[ABS(u)] = VS_FROZEN;
}
void k_parse_units(const DB& db, const u32* ulit, u32 n, u32* first, u32* win, u32* pos, void* tmp, u32* total,
                   u32* trail, u32* err, Stream* st) {
  fill_u32(total, 0, 1, st);
  if (!n) return;
  fill_u32(first, 0xFFFFFFFFu, (size_t)db.nvars + 1, st);
  KLAUNCH(parse_claim_k, grid_for(n, 256), 256, st, ulit, n, first);
  KLAUNCH(parse_settle_k, grid_for(n, 256), 256, st, ulit, n, first, win, err);
  scan_u32(win, pos, n, total, tmp, st);
  KLAUNCH(parse_trail_k, grid_for(n, 256), 256, st, db, ulit, n, win, pos, trail);
}
__global__ void iota_u32_k(u32* a, u64 n) {
  const u64 k = (u64)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) a[k] = (u32)k;
}
void iota_u32(u32* a, size_t n, Stream* st) {
  if (!n) return;
  KLAUNCH(iota_u32_k, grid_for(n, 256), 256, st, a, (u64)n);
}

// ---------------------------------------------------------------- ELS
// Binary implication graph over literals (equivalence.cpp:26-40, 92-139):
// a live clause (a, b) of two active variables gives a -> ... edges
// -a -> b and -b -> a.  Out-edges are a CSR (off, adj); the in-edges of l
// are the negations of the out-edges of -l (the graph is skew-symmetric).
PF_DEV bool els_binary(const DB& db, u32 c, u32& a, u32& b) {
  if (is_deleted(db, c) || csize(db, c) != 2) return false;
  const u32* l = clits(db, c);
  a = l[0], b = l[1];
  return !db.vstate[ABS(a)] && !db.vstate[ABS(b)];
}
__global__ void els_deg_k(DB db, u32* deg) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  u32 a, b;
  if (i < db.ncls && els_binary(db, db.c_off[i], a, b)) {
    atomicAdd(&deg[FLIP(a)], 1u);
    atomicAdd(&deg[FLIP(b)], 1u);
  }
}
__global__ void els_fill_k(DB db, const u32* off, u32* cur, u32* adj) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  u32 a, b;
  if (i < db.ncls && els_binary(db, db.c_off[i], a, b)) {
    adj[off[FLIP(a)] + atomicAdd(&cur[FLIP(a)], 1u)] = b;
    adj[off[FLIP(b)] + atomicAdd(&cur[FLIP(b)], 1u)] = a;
  }
}
void k_els_graph(const DB& db, u32* deg, u32* off, void* tmp, Stream* st) {
  const size_t n2 = 2 * (size_t)db.nvars + 2;
  fill_u32(deg, 0, n2, st);
  if (db.ncls) KLAUNCH(els_deg_k, grid_for(db.ncls, 256), 256, st, db, deg);
  scan_u32(deg, off, n2, off + n2, tmp, st);
}
void k_els_fill(const DB& db, const u32* off, u32* cur, u32* adj, Stream* st) {
  fill_u32(cur, 0, 2 * (size_t)db.nvars + 2, st);
  if (db.ncls) KLAUNCH(els_fill_k, grid_for(db.ncls, 256), 256, st, db, off, cur, adj);
}
// Trimming: a literal without remaining in-edges or out-edges is an SCC of
// its own.  alive[l] = 1 for active literals still in the graph; a removed
// literal is its own root.  The first frontier holds the literals that
// start with no in- or out-edge.
__global__ void els_trim_init_k(DB db, const u32* off, u32* alive, u32* indeg, u32* outdeg, u32* root, u32* front,
                                u32* nfront) {
  __shared__ u32 lw[NW];
  const u32 n2 = 2 * db.nvars + 2, first = (blockIdx.x * blockDim.x + threadIdx.x) * SIPT;
  u32 bits = 0;
#pragma unroll
  for (u32 t = 0; t < (u32)SIPT; t++) {
    const u32 l = first + t;
    if (l >= n2) break;
    const bool act = l >= 2 && !db.vstate[ABS(l)];
    const u32 out = off[l + 1] - off[l], in = off[FLIP(l) + 1] - off[FLIP(l)];
    indeg[l] = in;
    outdeg[l] = out;
    root[l] = l;
    alive[l] = act && in && out ? 1u : 0u;
    if (act && !(in && out)) bits |= 1u << t;
  }
  u32 k = block_reserve(bits, lw, nfront);
  while (bits) {
    const u32 t = __ffs(bits) - 1;
    bits &= bits - 1;
    front[k++] = first + t;
  }
}
PF_DEV void els_drop(u32 w, u32* alive, u32* root, u32* next, u32* nnext) {
  if (atomicCAS(&alive[w], 1u, 0u) == 1u) {
    root[w] = w;
    next[atomicAdd(nnext, 1u)] = w;
  }
}
__global__ void els_trim_k(const u32* front, u32 n, const u32* off, const u32* adj, u32* alive, u32* indeg,
                           u32* outdeg, u32* root, u32* next, u32* nnext) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const u32 v = front[k];
  for (u32 j = off[v]; j < off[v + 1]; j++) {  // out-neighbours lose an in-edge
    const u32 w = adj[j];
    if (atomicSub(&indeg[w], 1u) == 1u) els_drop(w, alive, root, next, nnext);
  }
  const u32 nv = FLIP(v);
  for (u32 j = off[nv]; j < off[nv + 1]; j++) {  // in-neighbours lose an out-edge
    const u32 u = FLIP(adj[j]);
    if (atomicSub(&outdeg[u], 1u) == 1u) els_drop(u, alive, root, next, nnext);
  }
}
void k_els_trim_init(const DB& db, const u32* off, u32* alive, u32* indeg, u32* outdeg, u32* root, u32* front,
                     u32* nfront, Stream* st) {
  fill_u32(nfront, 0, 1, st);
  KLAUNCH(els_trim_init_k, grid_for(2 * (size_t)db.nvars + 2, STILE), ST, st, db, off, alive, indeg, outdeg, root,
          front, nfront);
}
void k_els_trim(const u32* front, u32 n, const u32* off, const u32* adj, u32* alive, u32* indeg, u32* outdeg, u32* root,
                u32* next, u32* nnext, Stream* st) {
  if (!n) return;
  KLAUNCH(els_trim_k, grid_for(n, 256), 256, st, front, n, off, adj, alive, indeg, outdeg, root, next, nnext);
}
// Coloring over the literals that survive trimming (list[0..n)): forward
// minimum labels, then from each root (color == itself) backwards inside
// its color; the marked literals form the root's SCC, whose root is its
// smallest literal.
__global__ void els_alive_k(u32 n2, const u32* alive, u32* list, u32* n) {
  __shared__ u32 lw[NW];
  const u32 first = (blockIdx.x * blockDim.x + threadIdx.x) * SIPT;
  u32 bits = 0;
#pragma unroll
  for (u32 t = 0; t < (u32)SIPT; t++)
    if (first + t < n2 && alive[first + t]) bits |= 1u << t;
  u32 k = block_reserve(bits, lw, n);
  while (bits) {
    const u32 t = __ffs(bits) - 1;
    bits &= bits - 1;
    list[k++] = first + t;
  }
}
__global__ void els_color_init_k(const u32* list, u32 n, u32* color, u32* mark) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  color[list[k]] = list[k];
  mark[list[k]] = 0;
}
__global__ void els_fw_k(const u32* list, u32 n, const u32* off, const u32* adj, const u32* alive, u32* color,
                         u32* changed) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const u32 v = list[k], c = color[v];
  for (u32 j = off[v]; j < off[v + 1]; j++) {
    const u32 w = adj[j];
    if (alive[w] && c < color[w] && atomicMin(&color[w], c) > c) *changed = 1;
  }
}
__global__ void els_roots_k(const u32* list, u32 n, const u32* color, u32* mark) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n && color[list[k]] == list[k]) mark[list[k]] = 1;
}
__global__ void els_bw_k(const u32* list, u32 n, const u32* off, const u32* adj, const u32* alive, const u32* color,
                         u32* mark, u32* changed) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const u32 v = list[k];
  if (mark[v]) return;
  const u32 c = color[v];
  for (u32 j = off[v]; j < off[v + 1]; j++) {
    const u32 w = adj[j];
    if (alive[w] && mark[w] && color[w] == c) {
      mark[v] = 1;
      *changed = 1;
      return;
    }
  }
}
__global__ void els_take_k(const u32* list, u32 n, const u32* mark, const u32* color, u32* alive, u32* root) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const u32 v = list[k];
  if (mark[v]) {
    root[v] = color[v];
    alive[v] = 0;
  }
}
// degrees inside the literals still alive (all counted before any is
// dropped), then the next trimming frontier
__global__ void els_redeg_k(const u32* list, u32 n, const u32* off, const u32* adj, const u32* alive, u32* indeg,
                            u32* outdeg) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const u32 v = list[k];
  if (!alive[v]) return;
  u32 out = 0, in = 0;
  for (u32 j = off[v]; j < off[v + 1]; j++) out += alive[adj[j]];
  const u32 nv = FLIP(v);
  for (u32 j = off[nv]; j < off[nv + 1]; j++) in += alive[FLIP(adj[j])];
  indeg[v] = in;
  outdeg[v] = out;
}
__global__ void els_redrop_k(const u32* list, u32 n, const u32* indeg, const u32* outdeg, u32* alive, u32* root,
                             u32* front, u32* nfront) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const u32 v = list[k];
  if (alive[v] && !(indeg[v] && outdeg[v])) els_drop(v, alive, root, front, nfront);
}
void k_els_alive(u32 n2, const u32* alive, u32* list, u32* n, Stream* st) {
  fill_u32(n, 0, 1, st);
  KLAUNCH(els_alive_k, grid_for(n2, STILE), ST, st, n2, alive, list, n);
}
void k_els_color_init(const u32* list, u32 n, u32* color, u32* mark, Stream* st) {
  if (n) KLAUNCH(els_color_init_k, grid_for(n, 256), 256, st, list, n, color, mark);
}
void k_els_fw(const u32* list, u32 n, const u32* off, const u32* adj, const u32* alive, u32* color, u32* changed,
              Stream* st) {
  fill_u32(changed, 0, 1, st);
  if (n) KLAUNCH(els_fw_k, grid_for(n, 256), 256, st, list, n, off, adj, alive, color, changed);
}
void k_els_roots(const u32* list, u32 n, const u32* color, u32* mark, Stream* st) {
  if (n) KLAUNCH(els_roots_k, grid_for(n, 256), 256, st, list, n, color, mark);
}
void k_els_bw(const u32* list, u32 n, const u32* off, const u32* adj, const u32* alive, const u32* color, u32* mark,
              u32* changed, Stream* st) {
  fill_u32(changed, 0, 1, st);
  if (n) KLAUNCH(els_bw_k, grid_for(n, 256), 256, st, list, n, off, adj, alive, color, mark, changed);
}
void k_els_take(const u32* list, u32 n, const u32* mark, const u32* color, u32* alive, u32* root, Stream* st) {
  if (n) KLAUNCH(els_take_k, grid_for(n, 256), 256, st, list, n, mark, color, alive, root);
}
void k_els_redeg(const u32* list, u32 n, const u32* off, const u32* adj, u32* alive, u32* indeg, u32* outdeg,
                 u32* root, u32* front, u32* nfront, Stream* st) {
  fill_u32(nfront, 0, 1, st);
  if (!n) return;
  KLAUNCH(els_redeg_k, grid_for(n, 256), 256, st, list, n, off, adj, alive, indeg, outdeg);
  KLAUNCH(els_redrop_k, grid_for(n, 256), 256, st, list, n, indeg, outdeg, alive, root, front, nfront);
}
// representatives (equivalence.cpp:66-118): rep[l] = root of l's SCC, l
// for assumed variables, 0 for inactive literals; info[0] |= 1 when a
// literal and its negation share an SCC, info[1] counts substituted literals
// grid-stride over a bounded number of workgroups: the count takes one
// atomic per workgroup (a single counter serialises its atomics)
__device__ inline void block_count_add(u32 mine, u32* lw, u32* out) {
  u32 tot;
  block_excl_scan(mine, lw, &tot);
  if (threadIdx.x == 0 && tot) atomicAdd(out, tot);
}
__global__ void els_rep_k(DB db, const u32* root, u32* rep, u32* info) {
  __shared__ u32 lw[NW];
  const u32 n2 = 2 * db.nvars + 2;
  u32 subs = 0;
  for (u32 l = blockIdx.x * blockDim.x + threadIdx.x; l < n2; l += gridDim.x * blockDim.x) {
    const u32 v = ABS(l);
    if (l < 2 || db.vstate[v]) {
      rep[l] = 0;
      continue;
    }
    const u32 r = root[l];
    if (root[FLIP(l)] == r) atomicOr(&info[0], 1u);
    rep[l] = db.assumed[v] ? l : r;
    subs += rep[l] != l;
  }
  block_count_add(subs, lw, &info[1]);
}
void k_els_rep(const DB& db, const u32* root, u32* rep, u32* info, Stream* st) {
  KLAUNCH(els_rep_k, std::min(grid_for(2 * (size_t)db.nvars + 2, ST), RED_BLOCKS), ST, st, db, root, rep, info);
}
// the clauses a substitution touches, with their position in the order
// learnts, then originals (lrank: exclusive scan of the learnt flags)
__global__ void els_learnt_k(DB db, u32* flag) {
  const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < db.ncls) flag[i] = st_learnt(cflags(db, db.c_off[i])) && !is_deleted(db, db.c_off[i]) ? 1u : 0u;
}
// the clauses in order, a tile's neighbours read by neighbouring lanes (eight
// in a row per lane took 0.15 ms for 500,000 variables, this less than 0.09)
__global__ void __launch_bounds__(ST) els_touch_k(DB db, const u32* rep, const u32* lrank, u32 nlearnt, u32* list,
                                                  u32* pos, u32* n) {
  __shared__ u32 lw[NW], cnt[ST];
  __shared__ u32 base;
  const u32 first = blockIdx.x * STILE + threadIdx.x, wave = threadIdx.x >> 6;
  u64 hits[SIPT];
#pragma unroll
  for (int t = 0; t < SIPT; t++) {
    const u32 i = first + t * ST;
    bool hit = false;
    if (i < db.ncls) {
      const u32 c = db.c_off[i];
      if (!is_deleted(db, c)) {
        const u32* l = clits(db, c);
        const u32 sz = csize(db, c);
        for (u32 q = 0; q < sz && !hit; q++) hit = rep[l[q]] != l[q];
      }
    }
    hits[t] = __ballot(hit);
  }
  cnt[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < SIPT; t++)
    if ((threadIdx.x & 63) == 0) cnt[t * NW + wave] = (u32)__popcll(hits[t]);
  __syncthreads();
  u32 tot;
  const u32 pre = block_excl_scan(cnt[threadIdx.x], lw, &tot);
  cnt[threadIdx.x] = pre;
  if (threadIdx.x == 0) base = tot ? atomicAdd(n, tot) : 0u;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < SIPT; t++) {
    const u64 below = (1ull << (threadIdx.x & 63)) - 1;
    if (!((hits[t] >> (threadIdx.x & 63)) & 1)) continue;
    const u32 i = first + t * ST, c = db.c_off[i], k = base + cnt[t * NW + wave] + (u32)__popcll(hits[t] & below);
    list[k] = c;
    pos[k] = st_learnt(cflags(db, c)) ? lrank[i] : nlearnt + (i - lrank[i]);
  }
}
void k_els_touch(const DB& db, const u32* rep, u32* lrank, void* tmp, u32* nlearnt, u32* list, u32* pos, u32* n,
                 Stream* st) {
  fill_u32(n, 0, 1, st);
  fill_u32(nlearnt, 0, 1, st);
  if (!db.ncls) return;
  KLAUNCH(els_learnt_k, grid_for(db.ncls, 256), 256, st, db, lrank);
  scan_u32(lrank, lrank, db.ncls, nlearnt, tmp, st);
}
void k_els_touch_list(const DB& db, const u32* rep, const u32* lrank, u32 nlearnt, u32* list, u32* pos, u32* n,
                      Stream* st) {
  if (db.ncls) KLAUNCH(els_touch_k, grid_for(db.ncls, STILE), ST, st, db, rep, lrank, nlearnt, list, pos, n);
}
// one pass of the unit-time fixpoint: the unit each touched clause yields
// under the current times (ptime: 2 p + sign, the smallest position wins).
// A second kept literal ends a clause: 0.31 -> 0.14 ms for a pass over 500,000
// variables' touched clauses, which compared each literal with all before it
// (0.13 with the short ones in registers).
__global__ void els_check_k(DB db, const u32* list, const u32* pos, u32 n, ElsView e, u32* ptime) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  u32 u = 0, m = 0;
  if (els_clause(db, list[k], e, pos[k], false, &u, &m) == 3) atomicMin(&ptime[ABS(u)], 2 * pos[k] + SIGN(u));
}
__global__ void els_commit_k(u32 n1, const u32* ptime, u32* utime, u32* changed) {
  const u32 v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v < n1 && ptime[v] != utime[v]) {
    utime[v] = ptime[v];
    *changed = 1;
  }
}
void k_els_check(const DB& db, const u32* list, const u32* pos, u32 n, const ElsView& e, u32* ptime, Stream* st) {
  fill_u32(ptime, NOPOS, (size_t)db.nvars + 1, st);
  if (n) KLAUNCH(els_check_k, grid_for(n, 256), 256, st, db, list, pos, n, e, ptime);
}
void k_els_commit(u32 n1, const u32* ptime, u32* utime, u32* changed, Stream* st) {
  fill_u32(changed, 0, 1, st);
  KLAUNCH(els_commit_k, grid_for(n1, 256), 256, st, n1, ptime, utime, changed);
}
// the substitution itself; units as (position, literal) records; info[0]
// |= 1 on an empty clause, info[1] counts clauses rewritten to two literals
__global__ void els_apply_k(DB db, const u32* list, const u32* pos, u32 n, ElsView e, u32* ukey, u32* uval, u32* nu,
                            u32* info) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  u32 u = 0, m = 0;
  const u32 kind = els_clause(db, list[k], e, pos[k], true, &u, &m);
  if (kind == 2) atomicOr(&info[0], 1u);
  if (kind == 3) {
    const u32 r = atomicAdd(nu, 1u);
    ukey[r] = pos[k];
    uval[r] = u;
  }
  if (kind == 4 && m == 2) atomicAdd(&info[1], 1u);
}
void k_els_apply(const DB& db, const u32* list, const u32* pos, u32 n, const ElsView& e, u32* ukey, u32* uval, u32* nu,
                 u32* info, Stream* st) {
  fill_u32(nu, 0, 1, st);
  if (n) KLAUNCH(els_apply_k, grid_for(n, 256), 256, st, db, list, pos, n, e, ukey, uval, nu, info);
}
// units in position order onto the trail (enqueueUnit)
__global__ void els_enqueue_k(DB db, const u32* uval, u32 n, u32* trail) {
  const u32 k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const u32 u = uval[k];
  trail[k] = u;
  db.assign[ABS(u)] = u + 1;
  db.vstate[ABS(u)] = VS_FROZEN;
}
void k_els_enqueue(const DB& db, const u32* uval, u32 n, u32* trail, Stream* st) {
  if (n) KLAUNCH(els_enqueue_k, grid_for(n, 256), 256, st, db, uval, n, trail);
}
// substituted variables (equivalence.cpp:173-190): an active variable whose
// positive literal has another representative gets a binary record on the
// stack (MODEL::saveBinary, model.cpp:280-288) and, when the
// representative's variable is active, the state SUBSTITUTED
__global__ void els_subst_flags_k(DB db, const u32* rep, u32* flag) {
  const u32 v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v > db.nvars) return;
  flag[v] = v && !db.vstate[v] && rep[V2L(v)] != V2L(v) ? 1u : 0u;
}
__global__ void els_subst_k(DB db, const u32* rep, const u32* flag, const u32* pos, u32* stack, u32* nmarked) {
  __shared__ u32 lw[NW];
  u32 marked = 0;
  for (u32 v = blockIdx.x * blockDim.x + threadIdx.x; v <= db.nvars; v += gridDim.x * blockDim.x) {
    if (!flag[v]) continue;
    const u32 p = V2L(v), other = rep[p];
    u32* w = stack + 5 * (size_t)pos[v];
    w[0] = V2L(db.vorg[v]);
    w[1] = V2L(db.vorg[ABS(other)]) | SIGN(FLIP(other));
    w[2] = 2;
    w[3] = V2L(db.vorg[v]) | 1u;
    w[4] = 1;
    // the representative's variable is the smallest of its SCC, never marked here
    if (!db.vstate[ABS(other)]) {
      db.vstate[v] = VS_SUBSTITUTED;
      marked++;
    }
  }
  block_count_add(marked, lw, nmarked);
}
void k_els_subst_flags(const DB& db, const u32* rep, u32* flag, u32* pos, void* tmp, u32* total, Stream* st) {
  KLAUNCH(els_subst_flags_k, grid_for((size_t)db.nvars + 1, 256), 256, st, db, rep, flag);
  scan_u32(flag, pos, (size_t)db.nvars + 1, total, tmp, st);
}
void k_els_subst(const DB& db, const u32* rep, const u32* flag, const u32* pos, u32* stack, u32* nmarked,
                 Stream* st) {
  fill_u32(nmarked, 0, 1, st);
  KLAUNCH(els_subst_k, std::min(grid_for((size_t)db.nvars + 1, ST), RED_BLOCKS), ST, st, db, rep, flag, pos, stack,
          nmarked);
}

}  // namespace pfs
