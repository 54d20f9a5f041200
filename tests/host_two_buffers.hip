// Runs the ticket order of a persistent workgroup with two row buffers (mg_two_buffers.h)
// on the host, one thread a wave, with one wave late wherever it reads the shared ticket.
// Every wave must take the same tickets in the same order.  Built and run by
// test_host_checks.py with hipcc's host pass alone: nothing here touches a GPU.
#include "mg_two_buffers.h"

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>

constexpr int WAVES = 4;

// A barrier that gives up: waves that no longer agree would wait for ever.
struct Barrier {
  std::mutex mu;
  std::condition_variable cv;
  int waiting = 0;
  long turn = 0;
  void wait() {
    std::unique_lock<std::mutex> lock(mu);
    const long mine = turn;
    if (++waiting == WAVES) {
      waiting = 0;
      ++turn;
      cv.notify_all();
    } else if (!cv.wait_for(lock, std::chrono::seconds(10), [&] { return turn != mine; })) {
      printf("a wave waits at a barrier the others do not reach\n");
      fflush(stdout);
      _Exit(2);
    }
  }
};

struct Shared {
  std::atomic<unsigned> ticket{0}, epoch{0}, counter{0};
  Barrier barrier;
};

struct Wave {
  Shared& sh;
  int w, late, at;  // wave `late` is late at its read number `at`
  int reads = 0;
  void first() {
    if (w != 0) return;
    sh.ticket = sh.counter++;
    sh.epoch = 7;
  }
  unsigned next(unsigned) { return w == 0 ? sh.counter++ : 0u; }
  void share(unsigned t) {
    if (w == 0) sh.ticket = t;
  }
  unsigned ticket() {
    if (w == late && reads++ == at) std::this_thread::sleep_for(std::chrono::milliseconds(50));
    return sh.ticket;
  }
  unsigned epoch() { return sh.epoch; }
  void barrier() { sh.barrier.wait(); }
};

int main() {
  int bad = 0;
  for (unsigned chunks : {1u, 2u, 5u})
    for (int late = 0; late < WAVES; ++late)
      for (int at = 0; at < 3; ++at) {
        Shared sh;
        std::vector<unsigned> seen[WAVES], loaded[WAVES];
        std::vector<std::thread> waves;
        for (int w = 0; w < WAVES; ++w)
          waves.emplace_back([&, w] {
            Wave wave{sh, w, late, at};
            ew_two_buffers<unsigned>(
                wave, chunks, [&](unsigned t, unsigned& rows) { rows = t, loaded[w].push_back(t); },
                [&](unsigned t, unsigned e, unsigned& rows, auto&& mid) {
                  seen[w].push_back(e == 7 && rows == t ? t : ~0u);
                  mid();
                  wave.barrier();  // the carry's
                });
          });
        for (auto& t : waves) t.join();
        for (int w = 0; w < WAVES; ++w) {
          bool ok = seen[w].size() == chunks && loaded[w] == seen[w];
          for (unsigned i = 0; ok && i < chunks; ++i) ok = seen[w][i] == i;
          if (!ok) printf("chunks %u: wave %d went wrong, wave %d late at read %d\n", chunks, w,
                          late, at);
          bad += !ok;
        }
      }
  printf("%d waves wrong\n", bad);
  return bad != 0;
}
