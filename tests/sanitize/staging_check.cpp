// The library's transfers (dg-bgk_amd/csrc/staging.hpp) on a stand-in for the
// device: every size and direction gives the same bytes, and whichever copy
// or allocation fails, the error comes back, nothing still writes to the
// caller's arrays, and no pinned block that a copy may use is in the pool.
#include "staging.hpp"

#include <vector>

using namespace dgbgk;

#define CHECK(x)                                                     \
  do {                                                               \
    if (!(x)) {                                                      \
      std::fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #x);   \
      std::exit(1);                                                  \
    }                                                                \
  } while (0)

static stub::Stream stream;

static std::vector<char> bytes(size_t n, unsigned seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)((i + seed) * 2654435761u >> 13);
  return v;
}

// every block in the pool is idle
static void pool_idle() {
  std::vector<char*> b;
  const long before = stub::allocs;
  while (stub::allocs == before) b.push_back(StagePool::get().take());
  for (char* p : b) {
    CHECK(!p || !stub::used(p, kStageBlock));
    StagePool::get().give(p);
  }
}

static void reset(long fail_copy, long fail_alloc) {
  CHECK(hipStreamSynchronize(&stream) == hipSuccess);
  stub::copies = stub::allocs = 0;
  stub::fail_copy = fail_copy;
  stub::fail_alloc = fail_alloc;
}

static void copies(size_t n, bool toDev) {
  const auto want = bytes(n, (unsigned)n);
  for (long fail_alloc : {-1L, -2L, 1L}) {
    long made = 0;
    for (long fail = -1; fail <= made; fail += fail < 1 || fail + 2 >= made ? 1 : (made + 2) / 3) {
      std::vector<char> host = toDev ? want : std::vector<char>(n), dev(want);
      if (toDev) std::fill(dev.begin(), dev.end(), 0);
      reset(fail, fail_alloc);
      const hipError_t e = stage_copy(dev.data(), host.data(), n, toDev, &stream, 0);
      if (fail < 0) made = stub::copies;
      CHECK(!stub::used(host.data(), n) && !stub::used(dev.data(), n));
      CHECK((e == hipSuccess) == (fail < 0 || fail >= stub::copies));
      if (e == hipSuccess) CHECK(host == want && dev == want);
      reset(-1, -1);
      pool_idle();
    }
  }
}

static void fetches() {
  const auto dev = bytes(5000, 7);
  // two ranges as a batch's records that wrap, and rows with gaps in what is wanted
  for (int form = 0; form < 2; ++form)
    for (long fail_alloc : {-1L, -2L}) {
      long made = 0;
      for (long fail = -1; fail <= made; ++fail) {
        std::vector<char> out(3000);
        StagePart part[4] = {{dev.data() + 4000, out.data(), 1000}, {dev.data(), out.data() + 1000, 2000}};
        int parts = 2;
        if (form == 1) {
          parts = 4;
          for (int i = 0; i < 4; ++i)
            part[i] = {dev.data() + 700 * i, i == 2 ? nullptr : out.data() + 700 * i, 700};
        }
        reset(fail, fail_alloc);
        const hipError_t e = stage_fetch(part, parts, &stream);
        if (fail < 0) made = stub::copies;
        CHECK(!stub::used(out.data(), out.size()) && !stub::used(dev.data(), dev.size()));
        CHECK((e == hipSuccess) == (fail < 0 || fail >= stub::copies));
        if (e == hipSuccess)
          for (int i = 0; i < parts; ++i)
            if (part[i].host) CHECK(!std::memcmp(part[i].host, part[i].dev, part[i].n));
        reset(-1, -1);
        pool_idle();
      }
    }
}

// what a short-lived program pays for: a block is made once, and no more of
// them than pieces or than a transfer needs
static void few_blocks() {
  StagePool::get().user(-1);  // empties the pool
  StagePool::get().user(1);
  std::vector<char> a(3 * kStageBlock), b(a.size());
  reset(-1, -1);
  for (int i = 0; i < 3; ++i) CHECK(stage_copy(b.data(), a.data(), 100, true, &stream, 0) == hipSuccess);
  CHECK(stub::allocs == 1);
  CHECK(stage_copy(b.data(), a.data(), a.size(), true, &stream, 0) == hipSuccess);
  CHECK(stub::allocs == 1);
  CHECK(stage_copy(b.data(), a.data(), a.size(), false, &stream, 0) == hipSuccess);
  CHECK(stub::allocs <= 3);
}

int main() {
  StagePool::get().user(1);
  for (size_t n : {(size_t)1, kStageBlock - 1, kStageBlock, kStageBlock + 1, 3 * kStageBlock,
                   9 * kStageBlock + 5})
    for (bool toDev : {true, false}) copies(n, toDev);
  copies(kPageableIn + 5, true);
  few_blocks();
  fetches();
  StagePool::get().user(-1);
  CHECK(stub::live == 0);  // all given back with the last user
  std::puts("staging ok");
}
