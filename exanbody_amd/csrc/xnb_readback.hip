// xnb_readback.hip -- the caller's host memory to and from device arrays.
//
// A caller's buffers are ordinary (pageable) memory.  Copying each field straight into them,
// through the runtime's own staging and then, atom by atom, into the caller's layout, took 272
// ms for 8,388,608 particles and 0.26 ms for 500.  Here a kernel writes a chunk of particles in
// the caller's layout over the bus into a pinned block (57 GB/s) and the host copies it out
// while the next is on its way, from a certain size on with several threads (first touches
// of fresh destination pages bound one thread at 11-17 GB/s): 20 ms (39 GB/s) and 0.03 ms.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "xnb_readback.h"

namespace xnb_impl {

namespace {

// Pinned blocks shared by every context of the process.  At most kMaxBlocks exist; a reader
// that finds none free waits for one.  Idle blocks are freed with the last context.
constexpr size_t kHalfBytes = 1u << 20, kBlockBytes = 2 * kHalfBytes;
constexpr int kMaxBlocks = 32;
constexpr int kMaxWorkers = 8;
// Reads from here on use more than one thread.  Several threads that wait share CPUs until the
// scheduler spreads them, which takes up to 4 ms: 12 MB take 0.8-1.9 ms with one thread and
// 3.8-4.1 with eight, 49 MB 3.1-4.9 and 2.8-7.4, 190 MB 16.4 and 5.1, 780 MB 70 and 20.
constexpr size_t kThreadedBytes = 64u << 20;

struct Pool {
  std::mutex mu;
  std::condition_variable returned;
  char* idle[kMaxBlocks];
  int n_idle = 0, n_blocks = 0, n_ctx = 0;
};
Pool& pool() {
  static Pool* p = new Pool;  // never destroyed: contexts may outlive static destruction
  return *p;
}

void free_idle(Pool& P) {  // P.mu held
  while (P.n_idle > 0) {
    (void)hipHostFree(P.idle[--P.n_idle]);
    P.n_blocks--;
  }
}

struct Block {
  char* p = nullptr;
  // wait: for a block in use elsewhere, when the pool is at its bound or memory is short
  explicit Block(bool wait) {
    Pool& P = pool();
    std::unique_lock<std::mutex> lk(P.mu);
    for (;;) {
      if (P.n_idle > 0) {
        p = P.idle[--P.n_idle];
        return;
      }
      if (P.n_blocks < kMaxBlocks) {
        void* h = nullptr;
        if (hipHostMalloc(&h, kBlockBytes, hipHostMallocPortable | hipHostMallocCoherent) == hipSuccess) {
          P.n_blocks++;
          p = (char*)h;
          return;
        }
        (void)hipGetLastError();  // dealt with here: a later launch's check must not find it
        if (P.n_blocks == 0) return;
      }
      if (!wait) return;
      P.returned.wait(lk);
    }
  }
  ~Block() {
    if (!p) return;
    Pool& P = pool();
    std::lock_guard<std::mutex> lk(P.mu);
    P.idle[P.n_idle++] = p;
    if (P.n_ctx == 0) free_idle(P);
    P.returned.notify_one();
  }
  Block(const Block&) = delete;
  Block& operator=(const Block&) = delete;
};

int usable_cpus() {
  cpu_set_t set;
  if (sched_getaffinity(0, sizeof(set), &set) != 0) return 1;
  return std::max(1, CPU_COUNT(&set));
}

// Chunks of `per` of the n items, each at most half a block: launch(first, count, half) queues
// the chunk on the context's stream, sink(first, count, half) takes it once it has arrived.
// Both are called from several threads, each with a block of its own: while one half is copied
// out, the next chunk is on its way into the other.
template <class Launch, class Sink>
int read_chunks(xnb_ctx* c, size_t n, size_t per, size_t bytes, const Launch& launch, const Sink& sink) {
  if (n == 0) return XNB_OK;
  const size_t nchunks = (n + per - 1) / per;
  const int want = bytes < kThreadedBytes ? 1 : std::min({kMaxWorkers, usable_cpus(), (int)std::min<size_t>(nchunks, kMaxWorkers)});
  std::atomic<size_t> next{0};
  std::atomic<int> failed{(int)hipSuccess}, no_block{0};
  auto work = [&](bool first) {
    Block blk(first);  // the calling thread always gets one; the others only if one is to be had
    if (!blk.p) {
      if (first) no_block = 1;
      return;
    }
    hipEvent_t ev[2] = {nullptr, nullptr};
    hipError_t he = hipSetDevice(c->device);
    for (int h = 0; h < 2 && he == hipSuccess; h++) he = hipEventCreateWithFlags(&ev[h], hipEventDisableTiming);
    size_t at[2], m[2] = {0, 0};  // the chunk in each half; m 0: none
    int h = 0;
    auto put = [&](int k) {
      const size_t q = he == hipSuccess && failed == (int)hipSuccess ? next++ : nchunks;
      m[k] = 0;
      if (q >= nchunks) return;
      at[k] = q * per;
      m[k] = std::min(per, n - at[k]);
      he = launch(at[k], m[k], blk.p + (size_t)k * kHalfBytes);
      if (he == hipSuccess) he = hipEventRecord(ev[k], c->st);
    };
    for (put(h); he == hipSuccess && m[h] > 0; h ^= 1) {
      put(h ^ 1);
      if (he == hipSuccess) he = hipEventSynchronize(ev[h]);
      if (he == hipSuccess) sink(at[h], m[h], blk.p + (size_t)h * kHalfBytes);
    }
    if (he != hipSuccess) {
      failed = (int)he;
      (void)hipStreamSynchronize(c->st);  // nothing writes into the block once it is given back
    }
    for (int k = 0; k < 2; k++)
      if (ev[k]) (void)hipEventDestroy(ev[k]);
  };
  std::thread th[kMaxWorkers];
  int started = 0;
  try {
    while (started + 1 < want) {
      th[started] = std::thread(work, false);
      started++;
    }
  } catch (const std::exception&) {  // no thread, or no memory for one: the chunks go to those there are
  }
  work(true);
  for (int q = 0; q < started; q++) th[q].join();
  if (no_block) return fail(c, XNB_E_NOMEM, "pinned allocation failed");
  if (failed != (int)hipSuccess) return fail(c, XNB_E_HIP, std::string("read back: ") + hipGetErrorString((hipError_t)failed.load()));
  return XNB_OK;
}

}  // namespace

void readback_context_created() {
  Pool& P = pool();
  std::lock_guard<std::mutex> lk(P.mu);
  P.n_ctx++;
}

void readback_context_destroyed() {
  Pool& P = pool();
  std::lock_guard<std::mutex> lk(P.mu);
  if (--P.n_ctx == 0) free_idle(P);
}

int read_particles(xnb_ctx* c, bool ghosts, uint32_t* cell, double* r, double* v, double* f, double* ep, uint64_t* id, uint8_t* type) {
  const int fields = (r ? kPackR : 0) | (v ? kPackV : 0) | (f ? kPackF : 0) | (ep ? kPackE : 0) | (id ? kPackId : 0) |
                     (cell ? kPackCell : 0) | (type ? kPackType : 0);
  ghosts = ghosts && c->G > 0;
  const uint32_t n = c->N + (ghosts ? c->G : 0u);
  if (!fields) return XNB_OK;
  // Inner slots are in cell order already; ghost slots follow them, so with ghosts the order
  // over all cells is laid out first.
  const uint32_t* order = nullptr;
  if (ghosts) {
    int e;
    if ((e = scan(c, c->cell_n.p, c->g.ncells, 0, c->coff.p))) return e;
    launch_cell_order(n, c->slot_cell_A.p, c->cell_off.p, c->coff.p, c->plen.p, c->st);
    HIPCHK(c, hipGetLastError());
    order = c->plen.p;
  }
  const size_t each = pack_layout(kPackThreads, fields).bytes / kPackThreads;
  const size_t per = kHalfBytes / each / kPackThreads * kPackThreads;  // whole workgroups, so that sections stay aligned
  const PState A = c->A;
  const uint32_t* slot_cell = c->slot_cell_A.p;
  return read_chunks(
      c, n, per, (size_t)n * each,
      [&](size_t at, size_t m, char* blk) {
        void* d = nullptr;
        const hipError_t he = hipHostGetDevicePointer(&d, blk, 0);
        if (he != hipSuccess) return he;
        launch_pack_particles(A, slot_cell, order, (uint32_t)at, (uint32_t)m, fields, (char*)d, c->st);
        return hipGetLastError();
      },
      [&](size_t at, size_t m, const char* blk) {
        const PackLayout L = pack_layout((uint32_t)m, fields);
        if (r) std::memcpy(r + 3 * at, blk + L.r, 24 * m);
        if (v) std::memcpy(v + 3 * at, blk + L.v, 24 * m);
        if (f) std::memcpy(f + 3 * at, blk + L.f, 24 * m);
        if (ep) std::memcpy(ep + at, blk + L.ep, 8 * m);
        if (id) std::memcpy(id + at, blk + L.id, 8 * m);
        if (cell) std::memcpy(cell + at, blk + L.cell, 4 * m);
        if (type) std::memcpy(type + at, blk + L.type, m);
      });
}

int read_bytes(xnb_ctx* c, const void* src, size_t bytes, void* dst) {
  return read_chunks(
      c, bytes, kHalfBytes, bytes,
      [&](size_t at, size_t m, char* blk) { return hipMemcpyAsync(blk, (const char*)src + at, m, hipMemcpyDeviceToHost, c->st); },
      [&](size_t at, size_t m, const char* blk) { std::memcpy((char*)dst + at, blk, m); });
}

// The way in: the host gathers a chunk in slot order into half a block, field by field, and a
// kernel reads it over the bus (each word once, whole lines) while the next chunk is gathered.
// Needs no other host arrays than order and cell.
int write_particles(xnb_ctx* c, size_t n, const uint32_t* order, const uint32_t* cell, const double* r, const double* v,
                    const uint64_t* id, const uint8_t* type) {
  constexpr size_t per = kHalfBytes / kUnpackBytes;
  Block blk(true);
  if (!blk.p) return fail(c, XNB_E_NOMEM, "pinned allocation failed");
  hipEvent_t ev[2] = {nullptr, nullptr};
  hipError_t he = hipSuccess;
  for (int h = 0; h < 2 && he == hipSuccess; h++) he = hipEventCreateWithFlags(&ev[h], hipEventDisableTiming);
  int h = 0;
  for (size_t at = 0; at < n && he == hipSuccess; at += per, h ^= 1) {
    const size_t m = std::min(per, n - at);
    if (at >= 2 * per) he = hipEventSynchronize(ev[h]);
    if (he != hipSuccess) break;
    char* const half = blk.p + (size_t)h * kHalfBytes;
    double* const d = (double*)half;  // x, y, z, vx, vy, vz, id (u64), cell and type (u32 each): m of each
    uint64_t* const di = (uint64_t*)(d + 6 * m);
    uint32_t* const dc = (uint32_t*)(di + m);
    for (size_t t = 0; t < m; t++) {
      const size_t p = order[at + t];
      for (int a = 0; a < 3; a++) d[(size_t)a * m + t] = r[3 * p + a];
      for (int a = 0; a < 3; a++) d[(size_t)(3 + a) * m + t] = v ? v[3 * p + a] : 0.0;
      di[t] = id ? id[p] : (uint64_t)p;
      dc[t] = cell[p];
      dc[m + t] = type ? type[p] : 0u;
    }
    void* dev = nullptr;
    he = hipHostGetDevicePointer(&dev, half, 0);
    if (he != hipSuccess) break;
    launch_unpack_particles(c->g, c->A, c->slot_cell_A.p, (uint32_t)at, (uint32_t)m, (const char*)dev, c->st);
    he = hipGetLastError();
    if (he == hipSuccess) he = hipEventRecord(ev[h], c->st);
  }
  const hipError_t hs = hipStreamSynchronize(c->st);  // the block is given back
  for (int k = 0; k < 2; k++)
    if (ev[k]) (void)hipEventDestroy(ev[k]);
  if (he == hipSuccess) he = hs;
  if (he != hipSuccess) return fail(c, XNB_E_HIP, std::string("particle upload: ") + hipGetErrorString(he));
  return XNB_OK;
}

}  // namespace xnb_impl
