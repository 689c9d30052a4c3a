// devmem.hip -- kept device blocks, pinned blocks and streams (devmem.hpp).
#include "devmem.hpp"

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "plan.hpp"

namespace bddc {

namespace {

struct Block {
  void *p;
  size_t bytes;
  int dev;   // device it lies on; of pinned memory: current when handed out
  int used;  // problem that used it last
  bool pinned;
};

struct Keep {
  std::mutex m;
  int problem = 1;
  std::unordered_map<void *, Block> out;    // handed out
  std::vector<Block> idle, idle_pinned;     // kept
  std::map<int, size_t> idle_bytes, bound;  // per device
  std::vector<std::pair<int, hipStream_t>> streams;
};
Keep &keep() {
  static Keep *k = new Keep();  // never destroyed: outlives the HIP runtime's teardown order
  return *k;
}

int current_device() {
  int d = 0;
  if (hipGetDevice(&d) != hipSuccess) fatal("DEVICE_ALLOC", "no current device");
  return d;
}

// a device current for a scope
struct OnDevice {
  int before = -1;
  explicit OnDevice(int dev) {
    if (hipGetDevice(&before) != hipSuccess || before == dev || hipSetDevice(dev) != hipSuccess) before = -1;
  }
  ~OnDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

// the smallest kept block (of one device, or -1) that fits without wasting
// more than a quarter
int best_fit(const std::vector<Block> &v, size_t bytes, int dev) {
  int best = -1;
  for (int k = 0; k < (int)v.size(); k++)
    if ((dev < 0 || v[k].dev == dev) && v[k].bytes >= bytes && v[k].bytes <= bytes + bytes / 4 + 4096 &&
        (best < 0 || v[k].bytes < v[best].bytes))
      best = k;
  return best;
}

void *take(Keep &K, std::vector<Block> &v, int k, int dev) {
  Block b = v[k];
  v[k] = v.back();
  v.pop_back();
  b.used = K.problem;
  b.dev = dev;
  K.out[b.p] = b;
  return b.p;
}

// gives back the kept device blocks (of one device, or -1) that `gone` accepts
template <class F> void give_back(Keep &K, int dev, F gone) {
  size_t o = 0;
  for (Block &b : K.idle) {
    if ((dev < 0 || b.dev == dev) && gone(b)) {
      K.idle_bytes[b.dev] -= b.bytes;
      (void)hipFree(b.p);
    } else {
      K.idle[o++] = b;
    }
  }
  K.idle.resize(o);
}

}  // namespace

void *dev_alloc(size_t bytes) {
  const int dev = current_device();
  const size_t unit = bytes < ((size_t)1 << 20) ? 4096 : (size_t)1 << 21;
  bytes = (std::max<size_t>(bytes, 1) + unit - 1) / unit * unit;
  Keep &K = keep();
  std::lock_guard<std::mutex> lock(K.m);
  const int k = best_fit(K.idle, bytes, dev);
  if (k >= 0) {
    K.idle_bytes[dev] -= K.idle[k].bytes;
    return take(K, K.idle, k, dev);
  }
  void *p = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e != hipSuccess && K.idle_bytes[dev] > 0) {
    (void)hipGetLastError();
    give_back(K, dev, [](const Block &) { return true; });
    e = hipMalloc(&p, bytes);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();
    fatal("BDDCML_DEVICE", "hipMalloc of " + std::to_string(bytes) + " bytes failed: " + hipGetErrorString(e));
  }
  K.out[p] = Block{p, bytes, dev, K.problem, false};
  return p;
}

// the block handed out at p, no longer held by its user; false: none
static bool withdraw(Keep &K, void *p, Block &b) {
  std::lock_guard<std::mutex> lock(K.m);
  const auto it = K.out.find(p);
  if (it == K.out.end()) return false;
  b = it->second;
  K.out.erase(it);
  return true;
}

void dev_free(void *p) {
  if (!p) return;
  Keep &K = keep();
  Block b{};
  if (!withdraw(K, p, b)) {
    (void)hipFree(p);
    return;
  }
  // work that uses it runs on the block's device, whichever is current now
  OnDevice on(b.dev);
  (void)hipDeviceSynchronize();
  std::lock_guard<std::mutex> lock(K.m);
  size_t &bound = K.bound[b.dev];
  if (bound == 0) {
    size_t avail = 0, total = 0;
    if (hipMemGetInfo(&avail, &total) != hipSuccess) total = 0;
    bound = std::max<size_t>(total / 8, 1);
  }
  if (K.idle_bytes[b.dev] + b.bytes > bound) {
    (void)hipFree(p);
    return;
  }
  K.idle_bytes[b.dev] += b.bytes;
  K.idle.push_back(b);
}

void *pinned_alloc(size_t bytes) {
  const int dev = current_device();
  bytes = (std::max<size_t>(bytes, 1) + 4095) / 4096 * 4096;
  Keep &K = keep();
  std::lock_guard<std::mutex> lock(K.m);
  const int k = best_fit(K.idle_pinned, bytes, -1);
  if (k >= 0) return take(K, K.idle_pinned, k, dev);
  void *p = nullptr;
  const hipError_t e = hipHostMalloc(&p, bytes, hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    fatal("BDDCML_DEVICE", std::string("hipHostMalloc failed: ") + hipGetErrorString(e));
  }
  K.out[p] = Block{p, bytes, dev, K.problem, true};
  return p;
}

void pinned_free(void *p) {
  Keep &K = keep();
  Block b{};
  if (!p || !withdraw(K, p, b)) return;
  OnDevice on(b.dev);
  (void)hipDeviceSynchronize();
  std::lock_guard<std::mutex> lock(K.m);
  K.idle_pinned.push_back(b);
}

hipStream_t stream_get() {
  const int dev = current_device();
  Keep &K = keep();
  std::lock_guard<std::mutex> lock(K.m);
  for (size_t k = 0; k < K.streams.size(); k++)
    if (K.streams[k].first == dev) {
      const hipStream_t st = K.streams[k].second;
      K.streams.erase(K.streams.begin() + k);
      return st;
    }
  hipStream_t st = nullptr;
  const hipError_t e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
  if (e != hipSuccess) fatal("BDDCML_DEVICE", std::string("hipStreamCreate failed: ") + hipGetErrorString(e));
  return st;
}

void stream_put(hipStream_t st) {
  if (!st) return;
  if (hipStreamSynchronize(st) != hipSuccess) {  // a stream in error is not handed on
    (void)hipGetLastError();
    (void)hipStreamDestroy(st);
    return;
  }
  hipDevice_t dev = 0;
  if (hipStreamGetDevice(st, &dev) != hipSuccess) dev = current_device();
  Keep &K = keep();
  std::lock_guard<std::mutex> lock(K.m);
  if (K.streams.size() >= 16) (void)hipStreamDestroy(st);
  else K.streams.push_back({(int)dev, st});
}

void devmem_bytes(double &held, double &kept) {
  Keep &K = keep();
  std::lock_guard<std::mutex> lock(K.m);
  held = kept = 0.0;
  for (const auto &o : K.out) held += o.second.pinned ? 0.0 : (double)o.second.bytes;
  for (const Block &b : K.idle) kept += (double)b.bytes;
}

void devmem_end_of_problem(bool nothing_held) {
  Keep &K = keep();
  std::lock_guard<std::mutex> lock(K.m);
  give_back(K, -1, [&](const Block &b) { return nothing_held || b.used != K.problem; });
  size_t o = 0;
  for (Block &b : K.idle_pinned) {
    if (nothing_held || b.used != K.problem) (void)hipHostFree(b.p);
    else K.idle_pinned[o++] = b;
  }
  K.idle_pinned.resize(o);
  if (nothing_held) {
    for (auto &s : K.streams) (void)hipStreamDestroy(s.second);
    K.streams.clear();
  }
  K.problem++;
}

}  // namespace bddc
