// fib_stage.h -- host transfers of a handle.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

namespace {

// One array of a host transfer: its place in the device staging buffer, its
// bytes, and the caller's array.
struct HostPart {
  size_t off, bytes;
  void *host;
};

// Places of a call's arrays in the staging buffer, in order.
struct Parts {
  HostPart v[5];  // X, V, Xi, types, sides at most
  int n = 0;
  size_t used = 0;
  size_t add(size_t bytes, const void *host) {  // 0 bytes when not wanted
    const size_t off = used;
    if (host) {
      v[n++] = {off, bytes, const_cast<void *>(host)};
      used += (bytes + 15) & ~(size_t)15;
    }
    return off;
  }
};

// Staging of a handle's host transfers: a device buffer that holds all arrays
// of one call (it grows to the largest call and stays) and, for calls of more
// than SMALL bytes, LANES pinned chunks.
//
// A small call's arrays go as one copy, from or to a row of host memory: a
// copy costs 10 us whatever it moves, pinned memory would gain 1 us in 11 for
// 64 KiB and cost 100 us on the first call, and the lanes' threads cost 30 us
// or more each.  By one copy and by lanes: set_state of 2.2 MB 165 and 213 us,
// of 4.0 MB 268 and 250, of 8.1 MB 490 and 355; state of 2.0 MB 194 and 206, of
// 3.6 MB 410 and 233, of 7.3 MB 800 and 400.  A large call's
// arrays go in chunks through LANES lanes, a host thread and a pinned chunk
// each, so that the lanes empty or fill theirs while another's is on the bus.
// One thread moves 25 GB/s between warm pages and pinned memory and 12 into
// pages that the caller has not touched yet, the bus 55, and every copy costs
// some 20 us on its stream: chunks of 512 KiB take 3.2 ms for 56 MB, of 1 MiB
// 2.3, of 2 MiB 1.9, of 4 MiB 1.8; six lanes or a stream per lane gain 2 to
// 7 %.  2.1 M atoms: set_state 3.4 -> 1.9 ms (and no allocations), forces 7.0
// -> 3.3 ms, state 14.6 -> 5.3 ms; 4 k atoms: set_state 88 -> 43 us.
struct Stage {
  static constexpr size_t SMALL = 2u << 20, CHUNK_MIN = 256u << 10,
                          CHUNK_MAX = 2u << 20;
  static constexpr int LANES = 4;
  size_t chunk = CHUNK_MAX, least = 0;  // see fit()
  int device = 0;
  char *dev = nullptr, *pin = nullptr;
  size_t dev_cap = 0;
  std::vector<char> row;           // of a small call
  hipEvent_t ev[LANES] = {};       // the lane's copy has ended

  // Sizes for a handle whose largest instance has n atoms.  Two chunks hold an
  // (n,3) array: pinned memory is slow to come by, 0.3 ms per MiB on its first
  // use.  The first buffer holds forces and energies, so that calls for them
  // after a smaller first call do not allocate again.
  void fit(size_t n) {
    const size_t set = n * 4 * sizeof(double);
    chunk = std::min(std::max((set * 3 / 8 + 0xffff) & ~(size_t)0xffff, CHUNK_MIN), CHUNK_MAX);
    least = set + 4096;
  }
  // Room for a call of `bytes`; without pinned memory (pin == nullptr) the
  // copies take the caller's pages.
  hipError_t reserve(size_t bytes) {
    if (bytes > dev_cap) {
      if (dev) (void)hipFree(dev);
      dev = nullptr;
      dev_cap = 0;
      const size_t cap = std::max(bytes, std::max(CHUNK_MIN, least));
      hipError_t e = hipMalloc((void **)&dev, cap);
      if (e != hipSuccess) return e;
      dev_cap = cap;
    }
    if (bytes <= SMALL) return hipSuccess;
    if (!pin &&
        hipHostMalloc((void **)&pin, LANES * chunk, hipHostMallocDefault) != hipSuccess) {
      pin = nullptr;
      (void)hipGetLastError();
    }
    for (int k = 0; k < LANES; ++k)
      if (!ev[k]) {
        hipError_t e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
        if (e != hipSuccess) return e;
      }
    return hipSuccess;
  }
  void release() {
    if (dev) (void)hipFree(dev);
    if (pin) (void)hipHostFree(pin);
    for (auto &e : ev)
      if (e) (void)hipEventDestroy(e), e = nullptr;
    dev = pin = nullptr;
    dev_cap = 0;
  }

  // The arrays between the caller and `dev`, after what the stream holds: up
  // to the device (the caller's arrays are read when this returns, the copies
  // may still be on the stream) or back (complete).  Throws nothing, as its
  // callers are C functions: without host memory it fails, without a thread
  // the calling one takes the lane.
  hipError_t copy(bool up, const Parts &P, hipStream_t s) {
    size_t total = 0;
    for (int k = 0; k < P.n; ++k) total = std::max(total, P.v[k].off + P.v[k].bytes);
    bool direct = total > SMALL && pin == nullptr;
    for (int k = 0; k < P.n; ++k) {
      hipPointerAttribute_t at{};
      if (hipPointerGetAttributes(&at, P.v[k].host) != hipSuccess) (void)hipGetLastError();
      direct = direct || at.type == hipMemoryTypeDevice;
    }
    if (direct) return copy_direct(up, P, s);
    std::vector<HostPart> ch;
    try {
      if (total <= SMALL) row.resize(std::max(row.size(), total));
      else
        for (int k = 0; k < P.n; ++k)
          for (size_t o = 0; o < P.v[k].bytes; o += chunk)
            ch.push_back({P.v[k].off + o, std::min(chunk, P.v[k].bytes - o),
                          (char *)P.v[k].host + o});
    } catch (const std::bad_alloc &) {
      return hipErrorOutOfMemory;
    }
    if (total <= SMALL) return copy_row(up, P, total, s);
    std::atomic<int> bad{(int)hipSuccess};
    auto lane = [&](int w) {
      hipError_t e = hipSetDevice(device);
      if (e == hipSuccess) e = up ? lane_up(w, ch, s) : lane_back(w, ch, s);
      if (e != hipSuccess) bad = (int)e;
    };
    const int nl = (int)std::min<size_t>(LANES, ch.size());
    std::thread th[LANES];
    int started = 1;
    try {
      for (; started < nl; ++started) th[started] = std::thread(lane, started);
    } catch (...) {  // no thread to be had (or no memory for one)
    }
    int cur = device;
    (void)hipGetDevice(&cur);
    lane(0);
    for (int w = started; w < nl; ++w) lane(w);
    for (int w = 1; w < started; ++w) th[w].join();
    (void)hipSetDevice(cur);
    if (bad != (int)hipSuccess) (void)hipStreamSynchronize(s);  // nothing in flight in `pin`
    return (hipError_t)bad.load();
  }

 private:
  hipError_t copy_direct(bool up, const Parts &P, hipStream_t s) {
    for (int k = 0; k < P.n; ++k) {
      const HostPart &q = P.v[k];
      hipError_t e = up ? hipMemcpyAsync(dev + q.off, q.host, q.bytes, hipMemcpyHostToDevice, s)
                        : hipMemcpyAsync(q.host, dev + q.off, q.bytes, hipMemcpyDeviceToHost, s);
      if (e != hipSuccess) return e;
    }
    return hipStreamSynchronize(s);
  }
  hipError_t copy_row(bool up, const Parts &P, size_t total, hipStream_t s) {
    if (up)
      for (int k = 0; k < P.n; ++k)
        std::memcpy(row.data() + P.v[k].off, P.v[k].host, P.v[k].bytes);
    hipError_t e = up ? hipMemcpyAsync(dev, row.data(), total, hipMemcpyHostToDevice, s)
                      : hipMemcpyAsync(row.data(), dev, total, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess && !up) e = hipStreamSynchronize(s);
    if (e == hipSuccess && !up)
      for (int k = 0; k < P.n; ++k)
        std::memcpy(P.v[k].host, row.data() + P.v[k].off, P.v[k].bytes);
    return e;
  }
  // lane w takes chunks w, w + LANES, ..., through its pinned one
  hipError_t lane_up(int w, const std::vector<HostPart> &ch, hipStream_t s) {
    char *const slot = pin + (size_t)w * chunk;
    hipError_t e = hipSuccess;
    for (size_t c = w; e == hipSuccess && c < ch.size(); c += LANES) {
      if (c >= LANES) e = hipEventSynchronize(ev[w]);
      if (e != hipSuccess) break;
      std::memcpy(slot, ch[c].host, ch[c].bytes);
      e = hipMemcpyAsync(dev + ch[c].off, slot, ch[c].bytes, hipMemcpyHostToDevice, s);
      if (e == hipSuccess) e = hipEventRecord(ev[w], s);
    }
    return e;
  }
  hipError_t lane_back(int w, const std::vector<HostPart> &ch, hipStream_t s) {
    char *const slot = pin + (size_t)w * chunk;
    hipError_t e = hipSuccess;
    for (size_t c = w; e == hipSuccess && c < ch.size(); c += LANES) {
      e = hipMemcpyAsync(slot, dev + ch[c].off, ch[c].bytes, hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipEventRecord(ev[w], s);
      if (e == hipSuccess) e = hipEventSynchronize(ev[w]);
      if (e == hipSuccess) std::memcpy(ch[c].host, slot, ch[c].bytes);
    }
    return e;
  }
};

}  // namespace
