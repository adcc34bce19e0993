// transfer.hip -- FP64 per-node arrays between HBM and pageable host memory.
//
// Compiled with -ffp-contract=off (the shift arithmetic rounds as the plain
// conversion kernels' does).
//
// A host array that a program has just allocated is bound by its page faults
// (one thread writes 4.8 GB/s into fresh pages, eight 26-38 GB/s), and a copy
// into pageable memory through the runtime reaches 4 GB/s.  So a call takes a
// ring of pinned slots, kernels move the data between HBM and the slots in node
// order at the link's rate (53 GB/s to the host, 55 from it; conversion and
// layout cost nothing there), and a few threads move it between the slots and
// the caller's array, both sides running ahead of each other by half a ring.
// The ring stays with the domain, and then for the next one: the first touch of
// pinned memory costs up to 0.4 ms a MiB, and a ring made anew by each call paid it
// in every other one.  Slots of 512 KiB leave the link at 47 GB/s, 1 MiB (for 64
// MiB and more) at 50.
// Measured against copies plane by plane through the runtime: 400 steps of the
// porous channel 256 x 128 x 128 (layout "yzx") with rho and u read 215 -> 105
// ms, 300 MRT steps of 128^3 FP32 35.5 -> 20.2 ms, populations of 96^3 in and
// out 18.5 -> 9.3 ms.
//
// Threads live as long as the call.
#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "step_kernel.hpp"
#include "transfer.hpp"

namespace hlbm {

constexpr size_t MIB = (size_t)1 << 20;
constexpr size_t SLOT_SMALL = MIB / 2, SLOT_LARGE = MIB, LARGE_FROM = 64 * MIB;
constexpr int SLOTS = 16, THREADS = 8;
constexpr size_t BLOCK = SLOTS * SLOT_SMALL;  // one pinned allocation: the small slots, or half of the large ones
constexpr int BLOCKS = 2;
static_assert(BLOCKS * BLOCK == SLOTS * SLOT_LARGE, "large slots fill all blocks");

struct TransferRing {
  char* block[BLOCKS] = {};
  hipEvent_t ev[SLOTS] = {};
  int device = 0;
  bool sound = true;  // no transfer through it has failed
  ~TransferRing() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    for (char* b : block)
      if (b) (void)hipHostFree(b);
  }
  bool open() {
    if (hipGetDevice(&device) != hipSuccess || !pin(0)) return false;
    for (int k = 0; k < SLOTS; k++)
      if (hipEventCreateWithFlags(&ev[k], hipEventDisableTiming | hipEventReleaseToSystem) != hipSuccess) {
        ev[k] = nullptr;
        (void)hipGetLastError();
        return false;
      }
    return true;
  }
  // Large slots need the second block, which is pinned beside the first by the
  // first transfer that asks for them; without it the small ones serve on.
  size_t slot_bytes(bool large) { return large && pin(1) ? SLOT_LARGE : SLOT_SMALL; }
  // false after a reset of the device, which takes pinned memory with it
  bool alive() const {
    for (char* b : block) {
      hipPointerAttribute_t a;
      if (b && (hipPointerGetAttributes(&a, b) != hipSuccess || a.type != hipMemoryTypeHost)) {
        (void)hipGetLastError();
        return false;
      }
    }
    return true;
  }
  double* slot(int k, size_t bytes) const {
    const size_t per = BLOCK / bytes, i = (size_t)(k % SLOTS);
    return (double*)(block[i / per] + i % per * bytes);
  }

 private:
  bool pin(int b) {
    if (!block[b] && hipHostMalloc((void**)&block[b], BLOCK, hipHostMallocCoherent) != hipSuccess) {
      block[b] = nullptr;
      (void)hipGetLastError();
    }
    return block[b] != nullptr;
  }
};

// One ring per device waits for the next domain after its own was destroyed:
// its pinned pages cost 1 to 2 ms, which a program that makes a domain, reads it
// once and makes the next would pay each time (first read of new 44^3 FP64
// domains, populations 1.7 ms against 0.8 ms later).  At most 16 MiB a device,
// given back when SPARE_IDLE domains in a row have gone without large transfers.
constexpr int SPARE_IDLE = 8;
struct Spare {
  TransferRing* ring = nullptr;
  int idle = 0;
};
struct Spares {
  std::mutex mu;
  std::map<int, Spare> of;  // device -> spare
};
static Spares& spares() {
  static Spares* s = new Spares;  // never destroyed: the runtime may be gone by then
  return *s;
}

static TransferRing* take_ring() {
  int device = 0;
  if (hipGetDevice(&device) == hipSuccess) {
    std::lock_guard<std::mutex> l(spares().mu);
    const auto it = spares().of.find(device);
    if (it != spares().of.end() && it->second.ring) {
      TransferRing* r = it->second.ring;
      it->second = Spare{};
      if (r->alive()) return r;  // (else nothing of it is left to free)
    }
  }
  TransferRing* r = new TransferRing;
  if (r->open()) return r;
  delete r;
  return nullptr;
}

void return_ring(TransferRing* ring, int device) {
  TransferRing* drop = nullptr;
  try {
    std::lock_guard<std::mutex> l(spares().mu);
    Spare& s = spares().of[ring ? ring->device : device];
    if (ring && ring->sound && !s.ring) {
      s = Spare{ring, 0};
    } else if (ring) {
      drop = ring;
    } else if (s.ring && ++s.idle >= SPARE_IDLE) {
      drop = s.ring;
      s = Spare{};
    }
  } catch (const std::bad_alloc&) {
    drop = ring;
  }
  delete drop;
}

namespace {

// Below these sizes the runtime's own copies of whole planes are as fast (to the
// host 10 MiB 0.67 ms and 0.70 through the ring, 25 MiB 2.0 and 1.4; from warm
// host pages 25 MiB 1.3 either way, 38 MiB 1.9 and 1.6), unless every plane has
// to be rearranged on the host.  Populations read in the reference layout pay a
// little later than other rearranged planes: their rows are short copies for
// either (4.3 MiB 0.54 and 0.60-0.74, 6.8 MiB 0.73 and 0.67-0.79, 33 MiB 5.8 and
// 3.2).
constexpr size_t MIN_TO_HOST = 12 * MIB, MIN_TO_DEVICE = 32 * MIB;
constexpr size_t MIN_REARRANGED = 4 * MIB, MIN_REFERENCE_TO_HOST = 6 * MIB;

// node k of the host's order (x fastest) -> index in the device layout
struct NodeOrder {
  uint32_t nx, nxy;
  NodeDivisors div;
  NodeLayout lay;
};
template <bool PERM>
__device__ __forceinline__ uint32_t device_index(const NodeOrder& o, uint32_t k) {
  if constexpr (!PERM) {
    return k;
  } else {
    const uint32_t z = div_by(k, o.div.m01, o.div.s01), r = k - z * o.nxy;
    const uint32_t y = div_by(r, o.div.m0, o.div.s0);
    return node_at(o.lay, (int)(r - y * o.nx), (int)y, (int)z);
  }
}

// nodes [first, first + n) between a device plane and a slot; w + sig is the
// rest state of the plane's direction
template <class S, bool PERM>
__global__ void __launch_bounds__(256) k_export(const S* src, double* slot, uint32_t first, uint32_t n, NodeOrder o,
                                                double w, double sig) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const uint32_t j = device_index<PERM>(o, first + i);
  if constexpr (StoreOps<S>::shifted)
    slot[i] = (double)StoreOps<S>::ld(src, j) + (w + sig);
  else
    slot[i] = src[j];
}
template <class S, bool PERM>
__global__ void __launch_bounds__(256) k_import(S* dst, const double* slot, uint32_t first, uint32_t n, NodeOrder o,
                                                double w, double sig) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const uint32_t j = device_index<PERM>(o, first + i);
  if constexpr (StoreOps<S>::shifted)
    StoreOps<S>::st(dst, j, (float)(slot[i] - w - sig));
  else
    dst[j] = slot[i];
}

template <class S>
hipError_t move_t(bool out, void* dev, double* slot, uint32_t first, uint32_t n, const NodeOrder& o, bool perm,
                  double w, double sig, hipStream_t s) {
  const dim3 g((n + 255) / 256), b(256);
  if (out) {
    if (perm)
      hipLaunchKernelGGL((k_export<S, true>), g, b, 0, s, (const S*)dev, slot, first, n, o, w, sig);
    else
      hipLaunchKernelGGL((k_export<S, false>), g, b, 0, s, (const S*)dev, slot, first, n, o, w, sig);
  } else {
    if (perm)
      hipLaunchKernelGGL((k_import<S, true>), g, b, 0, s, (S*)dev, (const double*)slot, first, n, o, w, sig);
    else
      hipLaunchKernelGGL((k_import<S, false>), g, b, 0, s, (S*)dev, (const double*)slot, first, n, o, w, sig);
  }
  return hipGetLastError();
}

// Host side of a chunk: nodes [first, first + n) between the slot and a plane.
void copy_rows(const TransferGrid& g, bool out, double* slot, double* host, uint32_t first, uint32_t n) {
  if (!g.reference) {
    if (out)
      std::memcpy(host + first, slot, (size_t)n * 8);
    else
      std::memcpy(slot, host + first, (size_t)n * 8);
    return;
  }
  // the All box: two ghost layers per side
  const uint32_t nx = (uint32_t)g.n[0], ny = (uint32_t)g.n[1];
  const size_t Lx = nx + 4, Ly = ny + 4;
  for (uint32_t k = first; k < first + n;) {
    const uint32_t row = k / nx, x = k - row * nx, z = row / ny, y = row - z * ny;
    const uint32_t len = std::min(nx - x, first + n - k);
    double* h = host + ((size_t)(z + 2) * Ly + (y + 2)) * Lx + (x + 2);
    double* p = slot + (k - first);
    if (out)
      std::memcpy(h, p, (size_t)len * 8);
    else
      std::memcpy(p, h, (size_t)len * 8);
    k += len;
  }
}

struct Chunk {
  int plane;
  uint32_t first, n;
};

// Host-side copies of chunks 0, 1, 2, ..., done by a few threads as they are released.
class Copiers {
 public:
  template <class F>
  Copiers(int chunks, F&& job) : done_(chunks, 0), job_(std::forward<F>(job)) {}
  // false if not one thread could be started
  bool start(int threads) {
    try {
      for (int k = 0; k < threads; k++) pool_.emplace_back([this] { work(); });
    } catch (const std::system_error&) {
    }
    return !pool_.empty();
  }
  ~Copiers() {
    {
      std::lock_guard<std::mutex> l(mu_);
      stop_ = true;
    }
    todo_cv_.notify_all();
    for (auto& t : pool_) t.join();
  }
  // the next chunk may be copied
  void release_next() {
    {
      std::lock_guard<std::mutex> l(mu_);
      released_++;
    }
    todo_cv_.notify_one();
  }
  void wait(int c) {
    std::unique_lock<std::mutex> l(mu_);
    done_cv_.wait(l, [&] { return done_[c] != 0; });
  }

 private:
  void work() {
    for (;;) {
      int c;
      {
        std::unique_lock<std::mutex> l(mu_);
        todo_cv_.wait(l, [&] { return stop_ || taken_ < released_; });
        if (taken_ == released_) return;
        c = taken_++;
      }
      job_(c);
      {
        std::lock_guard<std::mutex> l(mu_);
        done_[c] = 1;
      }
      done_cv_.notify_one();
    }
  }
  std::mutex mu_;
  std::condition_variable todo_cv_, done_cv_;
  int released_ = 0, taken_ = 0;
  std::vector<char> done_;
  bool stop_ = false;
  std::function<void(int)> job_;
  std::vector<std::thread> pool_;
};

int transfer(TransferRing** owned, bool out, const TransferGrid& g, const NodePlane* planes, int count, hipStream_t s, hipError_t* err) {
  *err = hipSuccess;
  const uint32_t N = (uint32_t)g.n[0] * (uint32_t)g.n[1] * (uint32_t)g.n[2];
  const size_t total = (size_t)N * 8 * count;
  const bool perm = !(g.lay.ord[0] == 0 && g.lay.ord[1] == 1);
  const bool populations = planes[0].q >= 0;
  const size_t least = perm || g.reference ? (out && populations && !perm ? MIN_REFERENCE_TO_HOST : MIN_REARRANGED)
                                           : (out ? MIN_TO_HOST : MIN_TO_DEVICE);
  if (total < least) return TRANSFER_DECLINED;
  if (!*owned) *owned = take_ring();
  if (!*owned) return TRANSFER_DECLINED;
  TransferRing& ring = **owned;
  const size_t slot_bytes = ring.slot_bytes(total >= LARGE_FROM);
  const uint32_t per = (uint32_t)(slot_bytes / 8);
  constexpr int slots = SLOTS, ahead = SLOTS / 2;
  std::vector<Chunk> chunks;
  for (int p = 0; p < count; p++)
    for (uint32_t a = 0; a < N; a += per) chunks.push_back({p, a, std::min(per, N - a)});
  const int nc = (int)chunks.size();

  NodeOrder o;
  o.nx = (uint32_t)g.n[0];
  o.nxy = o.nx * (uint32_t)g.n[1];
  node_divisor(o.nx, o.div.m0, o.div.s0);
  node_divisor(o.nxy, o.div.m01, o.div.s01);
  o.lay = g.lay;

  auto slot = [&](int c) { return ring.slot(c, slot_bytes); };
  Copiers copiers(nc, [&](int c) {
    const Chunk& k = chunks[c];
    copy_rows(g, out, slot(c), planes[k.plane].host, k.first, k.n);
  });
  // about 2 MiB of copying pays for a thread
  if (!copiers.start((int)std::min<size_t>(THREADS, total >> 21))) return TRANSFER_DECLINED;

  auto device = [&](int c) -> hipError_t {
    const Chunk& k = chunks[c];
    const NodePlane& p = planes[k.plane];
    const double w = p.q < 0 ? 0.0 : WD(p.q), sig = p.q < 0 ? 0.0 : g.shift.s[dir_class(p.q)];
    hipError_t e = hipErrorInvalidValue;
    switch (p.q < 0 ? 0 : g.storage) {
      case 0: e = move_t<double>(out, p.dev, slot(c), k.first, k.n, o, perm, w, sig, s); break;
      case 1: e = move_t<float>(out, p.dev, slot(c), k.first, k.n, o, perm, w, sig, s); break;
      case 2: e = move_t<_Float16>(out, p.dev, slot(c), k.first, k.n, o, perm, w, sig, s); break;
      case 3: e = move_t<bf16s>(out, p.dev, slot(c), k.first, k.n, o, perm, w, sig, s); break;
    }
    return e == hipSuccess ? hipEventRecord(ring.ev[c % slots], s) : e;
  };
  auto landed = [&](int c) { return hipEventSynchronize(ring.ev[c % slots]); };

  hipError_t e = hipSuccess;
  if (out) {
    // chunk c's kernel is queued when the chunk that held its slot has been
    // copied out; chunk c - ahead is handed to the threads when it has landed
    for (int c = 0; c < nc + ahead && e == hipSuccess; c++) {
      if (c < nc) {
        if (c >= slots) copiers.wait(c - slots);
        e = device(c);
      }
      if (e == hipSuccess && c >= ahead) {
        e = landed(c - ahead);
        if (e == hipSuccess) copiers.release_next();
      }
    }
    if (e == hipSuccess)
      for (int c = std::max(0, nc - slots); c < nc; c++) copiers.wait(c);
  } else {
    // chunk c is filled when the kernel that read its slot has finished; chunk
    // c - ahead's kernel is queued when it has been filled
    for (int c = 0; c < nc + ahead && e == hipSuccess; c++) {
      if (c < nc) {
        if (c >= slots) e = landed(c - slots);
        if (e == hipSuccess) copiers.release_next();
      }
      if (e == hipSuccess && c >= ahead) {
        copiers.wait(c - ahead);
        e = device(c - ahead);
      }
    }
  }
  // nothing may still read or write the slots afterwards
  const hipError_t last = hipStreamSynchronize(s);
  *err = e != hipSuccess ? e : last;
  ring.sound = ring.sound && *err == hipSuccess;
  return *err == hipSuccess ? TRANSFER_DONE : TRANSFER_FAILED;
}

int guarded(TransferRing** ring, bool out, const TransferGrid& g, const NodePlane* planes, int count, hipStream_t s, hipError_t* err) {
  try {
    return transfer(ring, out, g, planes, count, s, err);
  } catch (const std::bad_alloc&) {  // before any work: the lists and threads come first
    *err = hipErrorOutOfMemory;
    return TRANSFER_FAILED;
  }
}

}  // namespace

int planes_to_host(TransferRing** ring, const TransferGrid& g, const NodePlane* planes, int count, hipStream_t s,
                   hipError_t* err) {
  return guarded(ring, true, g, planes, count, s, err);
}
int planes_to_device(TransferRing** ring, const TransferGrid& g, const NodePlane* planes, int count, hipStream_t s,
                     hipError_t* err) {
  return guarded(ring, false, g, planes, count, s, err);
}

}  // namespace hlbm
