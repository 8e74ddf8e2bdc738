// The host side of the photo uploads' pinned ring; no HIP in here.
#pragma once

#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace splat {

// Worker threads that copy a list of host images, cut into chunks, into the pinned ring in order;
// the calling thread hands each finished chunk to the GPU and frees ring slots as their copies end. A
// worker sleeps while the ring is full.
class RingFill {
 public:
  static constexpr size_t CHUNK = size_t(2) << 20;
  static constexpr int SLOTS = 8, THREADS = 3;  // one thread copies at about half the link's rate
  struct Chunk { const uint8_t* src; size_t bytes; };
  RingFill(uint8_t* ring, std::vector<Chunk> chunks) : ring_(ring), chunks_(std::move(chunks)), done_(chunks_.size()) {
    for (auto& d : done_) d.store(false, std::memory_order_relaxed);
    threads_.reserve(THREADS);
    try {
      for (int t = 0; t < THREADS && size_t(t) < chunks_.size(); ++t) threads_.emplace_back([this] { work(); });
    } catch (const std::exception&) {  // fewer threads than asked for: see help()
    }
  }
  ~RingFill() {
    {
      std::lock_guard<std::mutex> lock(mu_);
      stop_ = true;
    }
    room_.notify_all();
    for (auto& t : threads_) t.join();
  }
  size_t bytes(size_t i) const { return chunks_[i].bytes; }
  bool filled(size_t i) const { return done_[i].load(std::memory_order_acquire); }
  bool has_room(size_t i) {
    std::lock_guard<std::mutex> lock(mu_);
    return i < allowed_;
  }
  void free_one() {
    {
      std::lock_guard<std::mutex> lock(mu_);
      ++allowed_;
    }
    room_.notify_one();
  }
  // With no worker at all the calling thread copies the next chunk, if the ring has room.
  bool help() {
    if (!threads_.empty() || next_ >= chunks_.size() || next_ >= allowed_) return false;
    copy(next_++);
    return true;
  }

 private:
  void copy(size_t i) {
    std::memcpy(ring_ + (i % SLOTS) * CHUNK, chunks_[i].src, chunks_[i].bytes);
    done_[i].store(true, std::memory_order_release);
  }
  void work() {
    std::unique_lock<std::mutex> lock(mu_);
    while (true) {
      room_.wait(lock, [this] { return stop_ || next_ >= chunks_.size() || next_ < allowed_; });
      if (stop_ || next_ >= chunks_.size()) return;
      const size_t i = next_++;
      lock.unlock();
      copy(i);
      lock.lock();
    }
  }
  uint8_t* ring_;
  std::vector<Chunk> chunks_;
  std::vector<std::atomic<bool>> done_;
  std::mutex mu_;  // guards next_, allowed_ and stop_
  std::condition_variable room_;
  size_t next_ = 0, allowed_ = SLOTS;
  bool stop_ = false;
  std::vector<std::thread> threads_;
};

}  // namespace splat
