// The served form's host logic over hip_stub.cpp.  server_check PASSES: that many
// times 24 requests through one server, all of which finish.  server_check stall:
// a server whose device stops (STUB_STALL) fails every unfinished request with
// MA_ERR_DEVICE within its wait limit, refuses more, and can be destroyed.
// server_check pause: many passes with a limit of a second, for a process that is
// stopped and continued meanwhile.
// server_check threads: planning a request takes the server's setup thread alone.
#include <dirent.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <thread>
#include <vector>
#include "miniaero.h"

static double now() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}
static ma_options request(int i) {
  ma_options o;
  std::memset(&o, 0, sizeof o);
  const int m = 2 + i * 7 % 9;
  o.problem_type = 1;
  o.nx = 4 * m;
  o.ny = 2 * m;
  o.nz = m;
  o.lx = o.ly = o.lz = 1.0;
  o.dt = 1e-6;
  o.ntimesteps = 10 + i * 13 % 41;
  o.second_order_space = 1;
  o.viscous = i % 3 == 0;
  o.precision = MA_PRECISION_FP32;
  o.limiter = i % 3 == 1;
  return o;
}
#define CHECK(x)                                             \
  do {                                                       \
    if (!(x)) {                                              \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);    \
      std::fflush(stdout);                                   \
      std::_Exit(1);                                         \
    }                                                        \
  } while (0)

static int threads_here() {
  int n = 0;
  DIR* d = opendir("/proc/self/task");
  while (const dirent* e = readdir(d)) n += e->d_name[0] != '.';
  closedir(d);
  return n;
}

static int threads() {
  ma_server_config cfg = {600ll << 20, 1, 1, 0, 0};
  ma_server* S = nullptr;
  CHECK(ma_server_create(&cfg, &S) == MA_OK);
  std::atomic<bool> done{false};
  std::atomic<int> most{0};
  std::thread watch([&] {
    while (!done) most = std::max(most.load(), threads_here());
  });
  const int idle = threads_here();
  ma_options o = request(0);
  o.nx = 96;
  o.ny = 48;
  o.nz = 24;
  o.ntimesteps = 1;
  long long id = 0;
  CHECK(ma_server_submit(S, &o, &id) == MA_OK);
  ma_case_result r;
  const double t0 = now();
  while (ma_server_poll(S, &r, 1, 0.2) == 0) CHECK(now() - t0 < 60.0);
  CHECK(r.status == MA_OK);
  done = true;
  watch.join();
  std::printf("%d threads, at most %d while planning\n", idle, most.load());
  CHECK(most <= idle);
  ma_server_destroy(S);
  return 0;
}

int main(int argc, char** argv) {
  if (argc > 1 && !std::strcmp(argv[1], "threads")) return threads();
  const bool stall = argc > 1 && !std::strcmp(argv[1], "stall");
  const bool pause = argc > 1 && !std::strcmp(argv[1], "pause");
  const int passes = stall ? 1 : pause ? 1 << 30 : std::atoi(argv[1]);
  const double end = now() + 6.0;
  ma_server_config cfg = {600ll << 20, 16, 8, 0, 0};
  ma_server* S = nullptr;
  CHECK(ma_server_create(&cfg, &S) == MA_OK);
  CHECK(ma_server_set_wait_limit(S, 0.0) == MA_ERR_INVALID);
  CHECK(ma_server_set_wait_limit(S, stall ? 0.4 : pause ? 1.0 : 20.0) == MA_OK);
  int failed = 0;
  for (int p = 0; p < passes && (!pause || now() < end); ++p) {
    std::set<long long> ids;
    const double t0 = now();
    for (int i = 0; i < 24; ++i) {
      const ma_options o = request(i);
      long long id = 0;
      const ma_status st = ma_server_submit(S, &o, &id);
      CHECK(st == MA_OK || (stall && st == MA_ERR_DEVICE));
      if (!st) ids.insert(id);
    }
    while (!ids.empty()) {
      CHECK(now() - t0 < 20.0);
      ma_case_result r[64];
      const int n = ma_server_poll(S, r, 64, 0.2);
      CHECK(n >= 0);
      for (int k = 0; k < n; ++k) {
        CHECK(ids.erase(r[k].id) == 1);
        CHECK(r[k].status == MA_OK || (stall && r[k].status == MA_ERR_DEVICE));
        std::vector<double> U((size_t)r[k].cells * 5 + 5);
        CHECK(ma_server_get_state(S, r[k].id, U.data()) == r[k].status);
        failed += r[k].status != MA_OK;
        if (k % 2) CHECK(ma_server_release(S, r[k].id) == MA_OK);
      }
    }
  }
  CHECK(stall == (failed > 0));
  if (stall) {
    const ma_options o = request(0);
    long long id = 0;
    CHECK(ma_server_submit(S, &o, &id) == MA_ERR_DEVICE);
    std::printf("%s\n", ma_last_error());
  } else {  // some still running as the server goes
    for (int i = 0; i < 24; ++i) {
      const ma_options o = request(i);
      long long id = 0;
      CHECK(ma_server_submit(S, &o, &id) == MA_OK);
    }
  }
  const double t0 = now();
  ma_server_destroy(S);
  CHECK(now() - t0 < 10.0);
  std::printf("ok\n");
  std::fflush(stdout);
  std::_Exit(0);  // (threads that wait for a stopped device stay)
}
