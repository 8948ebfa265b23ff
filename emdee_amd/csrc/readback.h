// Vectors of doubles from the GPU to the caller's memory.
//
// The GPU writes them, chunk by chunk and already in the caller's order, into
// pinned host memory and posts a number after each chunk; the host copies a
// chunk on as soon as its number is there.  The caller's memory is pageable
// and one core moves about 15 GB/s, a third of what the GPU writes, so from
// READ_THREADED bytes on helper threads copy too.  They start when the first
// chunk has arrived (before, they would only wait for the work queued on the
// stream) and end before the call does.
// One copy into a staging buffer, a wait for it and a memcpy took 113, 217,
// 1,527 and 5,540 us for the three vectors of 12,288 atoms and the coordinates
// of 150,001, 1,048,576 and 4,194,304; this takes 77, 150, 615 and 2,230 (45
// GB/s; without helpers 1,060 and 3,990, with one 717 and 2,550, with seven as
// with three).  Chunks of a quarter of the vector, 0.5 to 2 MB: 450,003
// doubles in four chunks 152 us, in two 182, in one 203; 4 MB chunks are no
// faster for 100 MB.
#pragma once
#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace emdee {

constexpr size_t READ_CHUNK = 1 << 18, READ_CHUNK_MIN = 1 << 16;   // doubles
constexpr size_t READ_THREADED = 4u << 20;
constexpr int READ_HELPERS = 3;

struct ReadRing {
  const double* host;                            // pinned, coherent
  double* dev;                                   // its device address
  const volatile unsigned long long* seq;        // the last number posted
  size_t size;                                   // doubles
};

// n doubles to out.  push(first, count, to, number): queues the kernels that
// write elements first.. to `to` and then post `number`; wait(number): waits
// for it on the calling thread.  Chunk k's number is seq0 + k.
template <class Push, class Wait>
void read_back(double* out, size_t n, const ReadRing& ring, unsigned long long seq0, Push&& push, Wait&& wait) {
  const size_t chunk = std::min(ring.size, std::clamp(n / 4, READ_CHUNK_MIN, READ_CHUNK)), chunks = (n + chunk - 1) / chunk;
  const size_t slots = ring.size >= n ? chunks : ring.size / chunk;
  std::vector<std::atomic<size_t>> taken(std::min(slots, chunks));   // per slot: chunks copied on, the last one's index + 1
  for (auto& t : taken) t.store(0);
  std::atomic<size_t> next{ 0 };
  size_t queued = 0;
  auto feed = [&]() {
    while (queued < chunks && (queued < slots || taken[queued % slots].load(std::memory_order_acquire) + slots > queued)) {
      push(queued * chunk, std::min(chunk, n - queued * chunk), ring.dev + (queued % slots) * chunk, seq0 + queued);
      queued++;
    }
  };
  auto take = [&](size_t k) {
    memcpy(out + k * chunk, ring.host + (k % slots) * chunk, sizeof(double) * std::min(chunk, n - k * chunk));
    taken[k % slots].store(k + 1, std::memory_order_release);
  };
  auto help = [&]() {
    for (size_t k; (k = next.fetch_add(1)) < chunks;) {
      while (*ring.seq < seq0 + k) __builtin_ia32_pause();
      std::atomic_thread_fence(std::memory_order_acquire);
      take(k);
    }
  };
  feed();
  wait(seq0);
  std::vector<std::thread> helpers;
  if (sizeof(double) * n >= READ_THREADED) {
    const size_t most = std::min<size_t>({ (size_t)READ_HELPERS, chunks - 1, std::max(1u, std::thread::hardware_concurrency()) - 1u });
    try {
      for (size_t t = 0; t < most; t++) helpers.emplace_back(help);
    } catch (const std::system_error&) {         // no more threads: those that started, and this one
    }
  }
  for (size_t k; (k = next.fetch_add(1)) < chunks;) {
    do feed(); while (queued <= k);
    wait(seq0 + k);
    take(k);
  }
  while (queued < chunks) feed();
  for (std::thread& t : helpers) t.join();
}

}  // namespace emdee
