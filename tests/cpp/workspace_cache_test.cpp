// Host-only check of the library's per-(device, stream) workspace cache
// (credit_amd/csrc/workspace_cache.hpp) with a recording allocator: keying,
// growth, retirement (never freeing a pointer a caller may hold) and a
// failing allocation; and of the scratch that calls can do without: its bound,
// and one call at a time between its launches.  Built with g++ by
// tests/test_workspace_cache.py.
#include <stdio.h>
#include <stdlib.h>

#include <thread>
#include <vector>

#include "../../credit_amd/csrc/workspace_cache.hpp"

struct FakeAlloc {
  std::vector<size_t>* sizes;
  bool* fail;
  int operator()(int, void*, size_t bytes, char** out) const {
    if (*fail) return -6;
    sizes->push_back(bytes);
    *out = static_cast<char*>(malloc(bytes));
    return 0;
  }
};

#define CHECK(c)                                                   \
  do {                                                             \
    if (!(c)) {                                                    \
      fprintf(stderr, "FAILED line %d: %s\n", __LINE__, #c);       \
      return 1;                                                    \
    }                                                              \
  } while (0)

int stream_scratch() {
  std::vector<size_t> sizes;
  bool fail = true;
  credit::StreamScratch<FakeAlloc> scratch(4096, 3, FakeAlloc{&sizes, &fail});
  auto key = [](int i) { return reinterpret_cast<void*>(size_t{0x1000} * (i + 1)); };
  auto base = [&](int device, int i) { return scratch.use(device, key(i)).base; };
  // No memory: the call does without, and takes no pair's room.
  CHECK(base(0, 0) == nullptr && sizes.empty());
  fail = false;
  // One buffer of the one size per (device, stream), the same at every use.
  char *a = base(0, 0), *b = base(0, 1), *c = base(1, 0);
  CHECK(a != nullptr && b != nullptr && c != nullptr && a != b && a != c && b != c);
  CHECK(base(0, 0) == a && base(1, 0) == c);
  // Pairs past the bound go without, whatever the order: 3 buffers in all.
  for (int i = 2; i < 40; ++i) {
    const auto u = scratch.use(0, key(i));
    CHECK(u.base == nullptr && !u.lock.owns_lock());
  }
  CHECK(base(0, 1) == b && sizes == std::vector<size_t>(3, 4096));
  // Threads on one stream: the launches of one call are not parted by another's.
  std::vector<std::thread> ts;
  int inside = 0, most = 0, calls = 0;
  for (int t = 0; t < 8; ++t)
    ts.emplace_back([&] {
      for (int i = 0; i < 200; ++i) {
        const auto u = scratch.use(0, key(0));
        if (u.base != a) abort();
        ++inside;
        if (inside > most) most = inside;
        std::this_thread::yield();
        --inside;
        ++calls;
      }
    });
  for (auto& t : ts) t.join();
  CHECK(most == 1 && calls == 1600 && sizes.size() == 3);
  return 0;
}

int main() {
  std::vector<size_t> sizes;
  bool fail = false;
  credit::WorkspaceCache<FakeAlloc> cache(FakeAlloc{&sizes, &fail});
  void* s1 = reinterpret_cast<void*>(0x1000);
  void* s2 = reinterpret_cast<void*>(0x2000);
  char *a = nullptr, *b = nullptr, *c = nullptr, *d = nullptr;
  // Distinct (device, stream) keys get distinct buffers; the same key the same one.
  CHECK(cache.get(0, s1, 100, &a) == 0);
  CHECK(cache.get(0, s2, 100, &b) == 0);
  CHECK(cache.get(1, s1, 100, &c) == 0);
  CHECK(a != b && a != c && b != c);
  CHECK(cache.get(0, s1, 5000, &d) == 0 && d == a);  // fits the 1 MiB minimum
  CHECK(sizes.size() == 3 && sizes[0] == (size_t{1} << 20));
  CHECK(cache.peek(0, s2) == b && cache.peek(0, nullptr) == nullptr);
  CHECK(cache.capacity(0, s2) == (size_t{1} << 20) && cache.capacity(0, nullptr) == 0);
  // Growth: at least double, rounded to 1 MiB; the old buffer is retired, not freed.
  char* e = nullptr;
  CHECK(cache.get(0, s1, (size_t{1} << 20) + 1, &e) == 0);
  CHECK(e != a && sizes.back() == (size_t{2} << 20));
  CHECK(cache.retired_count() == 1);
  CHECK(cache.get(0, s1, (size_t{5} << 20) + 3, &e) == 0 && sizes.back() == (size_t{6} << 20));
  CHECK(cache.retired_count() == 2);
  a[0] = 1;  // still owned: a retired buffer stays valid for its holders
  // A failing allocation reports its status and keeps the old buffer.
  fail = true;
  char* f = nullptr;
  CHECK(cache.get(0, s1, size_t{64} << 20, &f) == -6 && f == nullptr);
  CHECK(cache.peek(0, s1) == e);
  fail = false;
  // Concurrent first use of one key from several threads yields one buffer.
  void* s3 = reinterpret_cast<void*>(0x3000);
  std::vector<char*> got(8, nullptr);
  std::vector<std::thread> ts;
  for (int i = 0; i < 8; ++i)
    ts.emplace_back([&, i] { cache.get(2, s3, 4096, &got[i]); });
  for (auto& t : ts) t.join();
  for (int i = 1; i < 8; ++i) CHECK(got[i] == got[0] && got[0] != nullptr);
  CHECK(cache.live().size() == 4);
  CHECK(stream_scratch() == 0);
  printf("workspace cache: ok\n");
  return 0;
}
