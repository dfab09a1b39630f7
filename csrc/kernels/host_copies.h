// Copies of some MB from host memory to host memory, by the caller and threads that help.
#pragma once
#include <pthread.h>
#include <string.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <new>
#include <thread>

// A host copy of some MB in pieces: a page comes out of memory, not of a cache, and one thread draws 24 to 33 GB/s.  Up to three threads
// help; they wait for copies of any caller, and end after two seconds without one (they are shared by a process: started for every copy
// they cost 15 to 20 us each).  Host memory to host memory, one thread / started for the copy / waiting: 1.5 MB 34 / 30 / 15 us, 3.5 MB 107 / 50 / 33, 8 MB
// 259 / 142 / 101.
// Nothing is thrown at the callers, who are C entries: where no memory or thread is to be had the caller copies by itself.
constexpr long COPY_PART = 640 << 10;
class CopyHelpers {
 public:
  static constexpr int MOST = 3;
  // A piece lies with its caller, who waits for it; `left` falls by one when it is over, and nothing of it is touched from then on.
  struct Piece {
    char* to;
    const char* from;
    long n;
    std::atomic<int>* left;
    Piece* next;
  };

  // Never ends: a helper may outlive the process's other objects.  A fork has none of its parent's threads and begins with its own.
  // Null without memory for it.
  static CopyHelpers* shared() {
    static std::atomic<CopyHelpers*> all{nullptr};
    static const int forks = pthread_atfork(nullptr, nullptr, [] { all.store(nullptr); });
    (void)forks;
    CopyHelpers* mine = all.load(std::memory_order_acquire);
    if (mine == nullptr) {
      CopyHelpers* const made = new (std::nothrow) CopyHelpers;
      if (made == nullptr || all.compare_exchange_strong(mine, made)) return made;
      delete made;
    }
    return mine;
  }
  // Queues the pieces; whatever no helper takes is taken by `finish`.
  void start(Piece* pieces, int n) {
    {
      std::lock_guard<std::mutex> hold(lock_);
      for (int i = 0; i < n; ++i) {
        pieces[i].next = nullptr;
        *end_ = &pieces[i];
        end_ = &pieces[i].next;
      }
      for (; helpers_ < MOST; ++helpers_) {
        try {
          std::thread([this] { help(); }).detach();
        } catch (...) {  // no thread to be had
          break;
        }
      }
    }
    ready_.notify_all();
  }
  void finish(const std::atomic<int>& left) {
    while (left.load(std::memory_order_acquire) > 0)
      if (!copy_one()) std::this_thread::yield();
  }

 private:
  bool copy_one() {
    std::unique_lock<std::mutex> hold(lock_);
    Piece* const p = first_;
    if (p == nullptr) return false;
    first_ = p->next;
    if (first_ == nullptr) end_ = &first_;
    hold.unlock();
    memcpy(p->to, p->from, p->n);
    p->left->fetch_sub(1, std::memory_order_release);
    return true;
  }
  void help() {
    for (;;) {
      if (copy_one()) continue;
      std::unique_lock<std::mutex> hold(lock_);
      if (!ready_.wait_for(hold, std::chrono::seconds(2), [this] { return first_ != nullptr; })) {
        --helpers_;
        return;
      }
    }
  }
  std::mutex lock_;
  std::condition_variable ready_;
  Piece *first_ = nullptr, **end_ = &first_;  // first come, first copied
  int helpers_ = 0;
};

// Pieces of a copy.
inline int copy_parts(long size) {
  const long parts = size / COPY_PART;
  return parts < 1 ? 1 : parts > CopyHelpers::MOST ? CopyHelpers::MOST + 1 : (int)parts;
}

// Over on return.
inline void copy_in_parts(char* to, const char* from, long size) {
  const int parts = copy_parts(size);
  CopyHelpers* const helpers = parts > 1 ? CopyHelpers::shared() : nullptr;
  if (helpers == nullptr) {
    memcpy(to, from, size);
    return;
  }
  const long each = size / parts & ~4095L;  // whole pages
  std::atomic<int> left{parts - 1};
  CopyHelpers::Piece pieces[CopyHelpers::MOST];
  for (int i = 0; i < parts - 1; ++i, to += each, from += each, size -= each) pieces[i] = {to, from, each, &left, nullptr};
  helpers->start(pieces, parts - 1);
  memcpy(to, from, size);
  helpers->finish(left);
}
