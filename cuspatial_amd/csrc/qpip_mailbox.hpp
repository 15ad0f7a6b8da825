// The list of pinned blocks that calls read their sizes back through (host code only).
#pragma once

#include <mutex>
#include <utility>
#include <vector>

namespace qpip {

// A block is lent to one call and given back when its stream has been waited for. A call
// that fails between its launch and the end of the wait sets the block aside: a kernel
// in flight may still write it, so it is not lent again, and trim frees it once the
// device that the kernel runs on has been waited for.
class MailboxList {
 public:
  // Null: none is free.
  void* take()
  {
    std::lock_guard<std::mutex> g(mu_);
    if (free_.empty()) return nullptr;
    void* const p = free_.back();
    free_.pop_back();
    return p;
  }
  void give(void* p)
  {
    std::lock_guard<std::mutex> g(mu_);
    free_.push_back(p);
  }
  void set_aside(void* p, int device)
  {
    std::lock_guard<std::mutex> g(mu_);
    aside_.emplace_back(p, device);
  }
  // Frees the free blocks, and those set aside on `device` if wait() says that it is idle.
  template <class Wait, class Free>
  void trim(int device, Wait wait, Free free_block)
  {
    std::lock_guard<std::mutex> g(mu_);
    for (void* p : free_) free_block(p);
    free_.clear();
    std::vector<std::pair<void*, int>> kept;
    bool const any = !aside_.empty();
    bool const idle = any && wait();
    for (auto const& [p, d] : aside_) {
      if (idle && d == device)
        free_block(p);
      else
        kept.emplace_back(p, d);
    }
    aside_.swap(kept);
  }

 private:
  std::mutex mu_;
  std::vector<void*> free_;
  std::vector<std::pair<void*, int>> aside_;
};

// One call's block. alloc() makes a new one or throws; device() is the caller's device.
class Mailbox {
 public:
  Mailbox(MailboxList& list, int (*device)(), void* (*alloc)())
    : list_(list), device_(device), p_(list.take())
  {
    if (!p_) p_ = alloc();
  }
  ~Mailbox()
  {
    try {
      if (in_flight_)
        list_.set_aside(p_, device_());
      else
        list_.give(p_);
    } catch (...) {  // no memory for the list's entry: the block stays allocated
    }
  }
  Mailbox(Mailbox const&)            = delete;
  Mailbox& operator=(Mailbox const&) = delete;
  void* get() const { return p_; }
  void launched() { in_flight_ = true; }
  void landed() { in_flight_ = false; }

 private:
  MailboxList& list_;
  int (*device_)();
  void* p_;
  bool in_flight_ = false;
};

}  // namespace qpip
