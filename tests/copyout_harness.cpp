// qs_copyout.hpp over a runtime of host memory whose calls can be made to fail: "fail=<call>:<n>"
// lets the n-th call of that name fail (n = 0: none), "bytes=<n>".  Copies four times and prints
// per copy: the result code, whether the data arrived, and how the runtime was used.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "qs_copyout.hpp"

static std::mutex mu;
static std::map<std::string, int> calls;
static std::string fail_name;
static int fail_at = 0, live_events = 0, live_buffers = 0, null_events = 0, waits_after_error = 0;
static bool failed(const char* name) {
  std::lock_guard<std::mutex> lk(mu);
  return ++calls[name] == fail_at && fail_name == name;
}

struct Fake {
  using Error = int;
  using Stream = int;
  using Event = int*;
  static constexpr int ok = 0;
  static int set_device(int) { return failed("set_device"); }
  static int host_alloc(void** p, size_t n) {
    if (failed("host_alloc")) return 1;
    live_buffers++;
    *p = malloc(n);
    return 0;
  }
  static void host_free(void* p) { live_buffers--; free(p); }
  static int event_create(int** e) {
    if (failed("event_create")) return 1;
    live_events++;
    *e = new int(0);
    return 0;
  }
  static void event_destroy(int* e) { live_events--; delete e; }
  static int event_record(int* e, int) {
    if (!e) { std::lock_guard<std::mutex> lk(mu); null_events++; return 2; }
    return failed("event_record");
  }
  static int event_wait(int*) { return failed("event_wait"); }
  static int stream_wait(int) { std::lock_guard<std::mutex> lk(mu); waits_after_error++; return 0; }
  static int copy(void* d, const void* s, size_t n, int) {
    if (failed("copy")) return 1;
    memcpy(d, s, n);
    return 0;
  }
  static void clear_error() {}
};

int main(int argc, char** argv) {
  size_t bytes = 0;
  for (int i = 1; i < argc; i++) {
    const std::string a = argv[i];
    if (a.rfind("bytes=", 0) == 0) bytes = strtoull(a.c_str() + 6, nullptr, 10);
    if (a.rfind("fail=", 0) == 0) {
      const size_t c = a.find(':');
      fail_name = a.substr(5, c - 5);
      fail_at = atoi(a.c_str() + c + 1);
    }
  }
  std::vector<unsigned char> src(bytes);
  {
    qs::CopyOut<Fake> out;
    for (int k = 0; k < 4; k++) {
      for (size_t i = 0; i < bytes; i++) src[i] = (unsigned char)((i * 2654435761u >> 13) + k);
      std::vector<unsigned char> dst(bytes);
      waits_after_error = 0;
      const int e = out.copy(0, dst.data(), src.data(), bytes, 0);
      printf("%d %d %d\n", e, dst == src ? 1 : 0, waits_after_error);
    }
  }
  printf("live %d %d null %d records %d\n", live_buffers, live_events, null_events, calls["event_record"]);
  return 0;
}
