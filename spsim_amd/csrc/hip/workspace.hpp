// The library workspace's bookkeeping: one buffer per device that every entry point
// without scratch memory of its own works in. Plain C++ over an Api of a few device
// calls, so that a host test can run it.
//
// Calls that use the buffer follow each other, whatever their threads and streams:
// a call holds the lock from its first look at the buffer until its work is
// enqueued, and the next one's stream waits on the device for an event behind the
// last one's work. The event takes 2.6 us of a stream's time (the 73 us of a small
// interpolated pattern became 75.5), so on a stream that never ends, where it can
// be recorded later, it is only recorded once another stream's call comes.
//
// A graph keeps the addresses that were captured: a buffer that a captured call was
// given outlives its replacement by a larger one, until release().
//
// Api: types Stream and Event, and static functions
//   bool alloc(void **, size_t), void free(void *), bool synchronize() (the device),
//   bool capturing(Stream), bool lasting(Stream) (it exists until the process ends,
//   and is never captured), bool record(Event *, Stream) (creates it first if it is
//   null), bool wait(Stream, Event)
#pragma once

#include <cstddef>
#include <mutex>
#include <new>

namespace spsim {

enum class WorkspaceResult { kOk, kNoMemory, kFailed };

template <class Api>
class SharedWorkspace {
 public:
  using Stream = typename Api::Stream;

  // The part of one call in the shared buffer; empty until acquire().
  class Use {
   public:
    explicit Use(Stream s) : s_(s) {}
    Use(const Use &) = delete;
    Use &operator=(const Use &) = delete;
    ~Use() { release(); }

    bool held() const { return ws_ != nullptr; }
    bool capturing() const { return capturing_; }

    // Takes the buffer for this call: waits for the calls before it. A stream that
    // is being captured neither waits nor records: what it captures runs when its
    // graph is launched.
    bool acquire(SharedWorkspace *ws) {
      if (ws_) return true;
      ws->mu_.lock();
      ws_ = ws;
      capturing_ = Api::capturing(s_);
      if (capturing_ || (ws->last_ == Last::kOpen && ws->open_ == s_)) return true;
      if (ws->last_ == Last::kOpen) ws->close(ws->open_);
      if (ws->last_ == Last::kOpen) return false;
      return ws->last_ == Last::kNone || Api::wait(s_, ws->done_);
    }

    bool holds(size_t bytes) const { return ws_->bytes_ >= bytes; }

    // At least `bytes` of the buffer, which is replaced by a larger one if it has to
    // grow (all work on the device has then ended).
    WorkspaceResult get(size_t bytes, void **ptr) {
      if (ws_->bytes_ < bytes) {
        if (!ws_->retire()) return WorkspaceResult::kFailed;
        void *p = nullptr;
        const size_t want = bytes + bytes / 4;
        if (!Api::alloc(&p, want)) return WorkspaceResult::kNoMemory;
        ws_->ptr_ = p;
        ws_->bytes_ = want;
      }
      *ptr = ws_->ptr_;
      used_ = true;
      ws_->captured_ = ws_->captured_ || capturing_;
      return WorkspaceResult::kOk;
    }

   private:
    void release() {
      if (!ws_) return;
      if (used_ && !capturing_) {
        ws_->last_ = Last::kOpen;
        ws_->open_ = s_;
        if (!Api::lasting(s_)) ws_->close(s_);
      }
      ws_->mu_.unlock();
      ws_ = nullptr;
    }
    Stream s_;
    SharedWorkspace *ws_ = nullptr;
    bool capturing_ = false, used_ = false;
  };

  // Frees the buffer, and those that graphs may still name.
  void release() {
    std::lock_guard<std::mutex> lk(mu_);
    captured_ = false;
    if (!retire()) return;
    while (kept_) {
      Kept *k = kept_;
      kept_ = k->next;
      Api::free(k->ptr);
      delete k;
    }
  }

 private:
  // The last call's work: none is left, it is all that open_ holds, or what done_ stands for.
  enum class Last { kNone, kOpen, kRecorded };

  // Records the event behind the work on s; without one, waits for it here.
  void close(Stream s) {
    if (Api::record(&done_, s))
      last_ = Last::kRecorded;
    else if (Api::synchronize())
      last_ = Last::kNone;
  }
  struct Kept {
    void *ptr;
    Kept *next;
  };

  // Leaves no buffer: it is freed, or kept if a graph may name it.
  bool retire() {
    if (!ptr_) return true;
    if (!Api::synchronize()) return false;
    if (!captured_)
      Api::free(ptr_);
    else if (Kept *k = new (std::nothrow) Kept{ptr_, kept_})  // without it the buffer stays until the process ends
      kept_ = k;
    ptr_ = nullptr;
    bytes_ = 0;
    captured_ = false;
    return true;
  }
  std::mutex mu_;
  void *ptr_ = nullptr;
  size_t bytes_ = 0;
  bool captured_ = false;
  Kept *kept_ = nullptr;
  Last last_ = Last::kNone;
  Stream open_{};
  typename Api::Event done_{};
};

}  // namespace spsim
