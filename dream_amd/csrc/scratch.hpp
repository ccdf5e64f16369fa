// scratch.hpp -- device buffers that threads keep between calls, and the
// allocations that may need their memory.
//
// A thread has one buffer per use, grown on demand.  It is busy from get to
// done; done says how many bytes may stay.  An idle buffer is given back when
// its thread ends or moves to another device, and -- any thread's -- when an
// allocation on its device fails, which is then tried once more.  Whoever
// calls done has waited for the stream, so an idle buffer is not in use on the
// device either.  `Memory` has current(), alloc(void **, size_t) and
// release(void *).
#pragma once

#include <algorithm>
#include <cstddef>
#include <mutex>
#include <vector>

namespace dream {

template <class Memory, int USES>
class ScratchPool {
public:
  struct Thread {
    int device = -1;
    void *p[USES] = {};
    size_t bytes[USES] = {};
    bool busy[USES] = {};
  };

  void join(Thread &t)
  {
    std::lock_guard<std::mutex> lock(mu_);
    threads_.push_back(&t);
  }
  void leave(Thread &t)
  {
    std::lock_guard<std::mutex> lock(mu_);
    threads_.erase(std::remove(threads_.begin(), threads_.end(), &t), threads_.end());
    for (int k = 0; k < USES; k++) drop(t, k);
  }

  // At least `bytes` for this use, or null.
  void *get(Thread &t, int use, size_t bytes)
  {
    std::lock_guard<std::mutex> lock(mu_);
    const int device = Memory::current();
    if (t.device != device) {
      for (int k = 0; k < USES; k++) drop(t, k);
      t.device = device;
    }
    t.busy[use] = true;
    bytes = std::max<size_t>(bytes, 1);
    if (t.bytes[use] >= bytes) return t.p[use];
    drop(t, use);
    const size_t want = (bytes + 65535) / 65536 * 65536;
    if (!Memory::alloc(&t.p[use], want) && !(give_back(device) && Memory::alloc(&t.p[use], want))) {
      t.p[use] = nullptr;
      t.busy[use] = false;
      return nullptr;
    }
    t.bytes[use] = want;
    return t.p[use];
  }
  void done(Thread &t, int use, size_t keep)
  {
    std::lock_guard<std::mutex> lock(mu_);
    t.busy[use] = false;
    if (t.bytes[use] > keep) drop(t, use);
  }

  // Any other allocation of the library.
  bool alloc(void **p, size_t bytes)
  {
    if (Memory::alloc(p, bytes)) return true;
    std::lock_guard<std::mutex> lock(mu_);
    return give_back(Memory::current()) && Memory::alloc(p, bytes);
  }

  // The same for an allocation made otherwise that failed: whether it may be
  // tried again.
  bool make_room()
  {
    std::lock_guard<std::mutex> lock(mu_);
    return give_back(Memory::current());
  }

private:
  static void drop(Thread &t, int k)
  {
    if (t.p[k]) Memory::release(t.p[k]);
    t.p[k] = nullptr;
    t.bytes[k] = 0;
  }
  bool give_back(int device)
  {
    bool any = false;
    for (Thread *t : threads_)
      for (int k = 0; k < USES; k++)
        if (t->device == device && !t->busy[k] && t->p[k]) {
          drop(*t, k);
          any = true;
        }
    return any;
  }

  std::mutex mu_;
  std::vector<Thread *> threads_;
};

} // namespace dream
