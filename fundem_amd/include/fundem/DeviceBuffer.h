// RAII device buffer owned by the host containers (the role of
// HostDeviceArray1D's device half, myHostDeviceArray.h:160-260). Allocation
// happens at set-up only; a step allocates nothing.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "../../../include/fundem_amd.h"

namespace fundem {

inline void hipCheck(hipError_t e, const char* what) {
  if (e != hipSuccess) {
    (void)hipGetLastError();  // do not leave the error for the next launch to report
    throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
  }
}

// A launcher's return code (FDM_OK or an error code) as an exception.
inline void fdmCheck(int r, const char* what) {
  if (r != FDM_OK) throw std::runtime_error(std::string(what) + " failed with code " + std::to_string(r));
}

template <class T>
class DeviceBuffer {
 public:
  DeviceBuffer() = default;
  ~DeviceBuffer() { release(); }
  DeviceBuffer(const DeviceBuffer&) = delete;
  DeviceBuffer& operator=(const DeviceBuffer&) = delete;
  DeviceBuffer(DeviceBuffer&& o) noexcept : p_(o.p_), n_(o.n_) {
    o.p_ = nullptr;
    o.n_ = 0;
  }
  DeviceBuffer& operator=(DeviceBuffer&& o) noexcept {
    if (this != &o) {
      release();
      p_ = o.p_;
      n_ = o.n_;
      o.p_ = nullptr;
      o.n_ = 0;
    }
    return *this;
  }

  // Resize without preserving contents; zero-filled when requested.
  void allocate(size_t n, bool zero = true) {
    if (n == n_ && p_) {
      if (zero) hipCheck(hipMemset(p_, 0, n_ * sizeof(T)), "hipMemset");
      return;
    }
    release();
    if (n > 0) {
      hipCheck(hipMalloc(&p_, n * sizeof(T)), "hipMalloc");
      n_ = n;
      if (zero) hipCheck(hipMemset(p_, 0, n_ * sizeof(T)), "hipMemset");
    }
  }
  void upload(const T* host, size_t n, hipStream_t s) {
    if (n > n_) allocate(n, false);
    if (n) hipCheck(hipMemcpyAsync(p_, host, n * sizeof(T), hipMemcpyHostToDevice, s), "upload");
  }
  void upload(const std::vector<T>& v, hipStream_t s) { upload(v.data(), v.size(), s); }
  void download(T* host, size_t n, hipStream_t s) const {
    if (n) hipCheck(hipMemcpyAsync(host, p_, n * sizeof(T), hipMemcpyDeviceToHost, s), "download");
  }
  std::vector<T> toHost(hipStream_t s, size_t n = (size_t)-1) const {
    if (n == (size_t)-1) n = n_;
    std::vector<T> h(n);
    download(h.data(), n, s);
    hipCheck(hipStreamSynchronize(s), "hipStreamSynchronize");
    return h;
  }
  void release() {
    if (p_) (void)hipFree(p_);
    p_ = nullptr;
    n_ = 0;
  }
  T* get() const { return p_; }
  size_t size() const { return n_; }
  double memoryGB() const { return double(n_ * sizeof(T)) / 1073741824.0; }

 private:
  T* p_ = nullptr;
  size_t n_ = 0;
};

// Pinned host memory that the process keeps between uses: freeing such a block
// slows the next copies and frees of the device's memory by up to 0.7 ms each
// (the life of a solver of 1500 bodies 14.5 -> 15.2 ms when each solver had
// its own). A block is given back as soon as nothing is in flight; at most
// kIdle blocks stay, the largest ones. Any thread and device may take one.
class PinnedPool {
 public:
  struct Block {
    double* p = nullptr;
    size_t words = 0;
  };
  static PinnedPool& get() {
    static PinnedPool* pool = new PinnedPool;  // (left to the process's end: the HIP runtime may go first)
    return *pool;
  }
  Block take(size_t words) {
    words = words < kLeast ? kLeast : words;
    {
      std::lock_guard<std::mutex> lock(m_);
      size_t best = idle_.size();
      for (size_t i = 0; i < idle_.size(); ++i)
        if (idle_[i].words >= words && (best == idle_.size() || idle_[i].words < idle_[best].words)) best = i;
      if (best < idle_.size()) {
        const Block b = idle_[best];
        idle_.erase(idle_.begin() + best);
        return b;
      }
    }
    Block b;
    hipCheck(hipHostMalloc((void**)&b.p, words * sizeof(double), hipHostMallocPortable), "hipHostMalloc");
    b.words = words;
    return b;
  }
  void give(Block b) {
    {
      std::lock_guard<std::mutex> lock(m_);
      if (idle_.size() < kIdle) {
        idle_.push_back(b);
        return;
      }
      for (auto& i : idle_)
        if (i.words < b.words) std::swap(i, b);
    }
    (void)hipHostFree(b.p);
  }
  static constexpr size_t kIdle = 4, kLeast = size_t(1) << 17;

 private:
  PinnedPool() { idle_.reserve(kIdle); }
  std::mutex m_;
  std::vector<Block> idle_;
};

}  // namespace fundem
