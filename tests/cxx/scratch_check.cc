// The scratch pool (scratch.hpp) on a memory of 10 blocks of 64 KiB per device:
// what is given back when an allocation fails, what is not, and threads.
// Prints the number of checks that failed.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>
#include <thread>

#include "scratch.hpp"

static thread_local int t_device = 0;
static std::mutex mem_mu;
static std::map<void *, std::pair<int, size_t>> live;     // device, bytes
static size_t used[2];
static std::atomic<int> wrong{0};
static const size_t kBlock = 65536, kAll = 10 * kBlock;

struct FakeMemory {
  static int current() { return t_device; }
  static bool alloc(void **p, size_t n)
  {
    std::lock_guard<std::mutex> lock(mem_mu);
    if (used[t_device] + n > kAll) return false;
    *p = std::malloc(n);
    live[*p] = {t_device, n};
    used[t_device] += n;
    return true;
  }
  static void release(void *p)
  {
    std::lock_guard<std::mutex> lock(mem_mu);
    auto it = live.find(p);
    if (it == live.end()) { wrong++; return; }
    used[it->second.first] -= it->second.second;
    live.erase(it);
    std::free(p);
  }
};
using Pool = dream::ScratchPool<FakeMemory, 3>;
static const size_t kKeep = 7 * kBlock;

static void check(bool ok, const char *what)
{
  if (!ok) { wrong++; std::fprintf(stderr, "failed: %s\n", what); }
}

int main()
{
  {
    Pool pool;
    Pool::Thread a, b;
    pool.join(a);
    pool.join(b);
    // Grown on demand, kept and served again.
    void *p = pool.get(a, 0, 5 * kBlock + 1);
    check(p && a.bytes[0] == 6 * kBlock, "rounded up");
    pool.done(a, 0, kKeep);
    check(pool.get(a, 0, 100) == p, "served again");
    // Busy buffers stay, whoever asks.
    check(!pool.get(b, 1, 8 * kBlock) && !b.busy[1], "no room beside a busy buffer");
    void *q = nullptr;
    check(!pool.alloc(&q, 8 * kBlock) && a.p[0] == p, "an allocation does not take it either");
    // Idle ones make room: for another thread, another use, another allocation.
    pool.done(a, 0, kKeep);
    check(pool.get(b, 1, 8 * kBlock) && !a.p[0], "idle scratch of another thread is given back");
    pool.done(b, 1, kKeep);
    check(!b.p[1] && used[0] == 0, "more than is kept goes at once");
    check(pool.get(a, 2, 6 * kBlock) != nullptr, "another use");
    pool.done(a, 2, kKeep);
    check(pool.get(a, 1, 3 * kBlock) && pool.get(a, 0, 5 * kBlock) && !a.p[2] && a.p[1],
          "an idle use of the same call's thread is given back, the busy one not");
    pool.done(a, 0, kKeep);
    check(pool.alloc(&q, 6 * kBlock) && !a.p[0] && a.p[1], "another allocation");
    FakeMemory::release(q);
    pool.done(a, 1, kKeep);
    check(pool.make_room() && used[0] == 0 && !pool.make_room(), "room made once");
    // Another device: this thread's buffers of the former one go, others' stay.
    check(pool.get(a, 0, kBlock) && pool.get(b, 0, 2 * kBlock), "both");
    pool.done(a, 0, kKeep);
    pool.done(b, 0, kKeep);
    t_device = 1;
    check(pool.get(a, 0, 9 * kBlock) && used[0] == 2 * kBlock, "moved");
    check(!pool.alloc(&q, 2 * kBlock) && b.p[0], "another device's idle scratch makes no room");
    t_device = 0;
    pool.leave(a);
    pool.leave(b);
    check(live.empty() && used[0] == 0 && used[1] == 0, "given back at the end");
  }
  {
    // Threads that fill their buffers while others' failures take idle ones.
    Pool pool;
    std::vector<std::thread> ts;
    std::atomic<int> served{0};
    for (int t = 0; t < 4; t++)
      ts.emplace_back([&, t]() {
        Pool::Thread me;
        pool.join(me);
        std::mt19937 gen((unsigned) t);
        for (int k = 0; k < 3000; k++) {
          const int use = (int) (gen() % 3);
          const size_t n = 1 + gen() % (4 * kBlock);
          unsigned char *p = (unsigned char *) pool.get(me, use, n);
          if (!p) continue;
          served++;
          p[0] = p[n - 1] = (unsigned char) (t + 1);
          std::this_thread::yield();
          if (p[0] != t + 1 || p[n - 1] != t + 1) wrong++;
          pool.done(me, use, 2 * kBlock);
        }
        pool.leave(me);
      });
    for (auto &t : ts) t.join();
    check(served > 3000, "served");
    check(live.empty(), "given back by the threads");
  }
  std::printf("%d\n", wrong.load());
  return 0;
}
