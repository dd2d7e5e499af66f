// The staged host transfers on a stand-in runtime (hip_stub): one named check
// per run, "ok" on success.
#include <dlfcn.h>
#include <fcntl.h>
#include <pthread.h>
#include <sys/stat.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <string>
#include <thread>
#include <vector>

#include "../critic2_amd/csrc/common.hpp"

using namespace c2;

// thread creation that fails after `threads_left` successes, and counts
static std::atomic<int> threads_left{-1}, threads_made{0};
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
  using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
  static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
  if (threads_left == 0) return EAGAIN;
  if (threads_left > 0) threads_left--;
  threads_made++;
  return real(t, a, f, x);
}

static void require(bool ok, const char *what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  std::exit(1);
}
#define REQUIRE(x) require((x), #x)

struct Ctx : c2gpu_ctx {
  Ctx() { stream = new stub::Stream; }
  ~Ctx() {
    release_stage(this);
    delete stream;
  }
};

static std::vector<char> bytes(size_t n, unsigned seed) {
  std::vector<char> v(n + 8);
  uint64_t x = seed * 2654435761u + 88172645463325252ull;
  for (size_t q = 0; q < n; q += 8) {
    x ^= x << 13;
    x ^= x >> 7;
    x ^= x << 17;
    std::memcpy(&v[q], &x, 8);
  }
  v.resize(n);
  return v;
}

constexpr size_t MIB = (size_t)1 << 20;
static const size_t SIZES[] = {1, 2 * MIB, 7 * MIB - 1, 7 * MIB, 7 * MIB + 3, 16 * MIB - 1, 16 * MIB, 26 * MIB - 7};

static void round_trip(c2gpu_ctx *ctx, size_t n, unsigned seed) {
  const std::vector<char> want = bytes(n, seed);
  std::vector<char> src = want, dev(n), dst(n);
  copy_in(ctx, dev.data(), src.data(), n);
  std::fill(src.begin(), src.end(), 0);  // pageable: it may change now
  (void)hipStreamSynchronize(ctx->stream);
  REQUIRE(dev == want);
  copy_out(ctx, dst.data(), dev.data(), n);
  std::fill(dev.begin(), dev.end(), 0);
  REQUIRE(dst == want);
}

static int temp_file() {
  char name[] = "/tmp/hostcopy_XXXXXX";
  const int fd = mkstemp(name);
  REQUIRE(fd >= 0);
  unlink(name);
  return fd;
}

static void file_trip(c2gpu_ctx *ctx, size_t n, unsigned seed) {
  const std::vector<char> want = bytes(n, seed);
  std::vector<char> dev = want, back(n);
  const int fd = temp_file();
  file_out(ctx, fd, 100, dev.data(), n);
  struct stat st;
  REQUIRE(fstat(fd, &st) == 0 && (size_t)st.st_size == 100 + n);
  file_in(ctx, back.data(), fd, 100, n, "short read");
  (void)hipStreamSynchronize(ctx->stream);
  REQUIRE(back == want);
  close(fd);
}

template <class F>
static int code_of(F &&f) {
  try {
    f();
  } catch (const Error &e) {
    return e.code;
  }
  return C2GPU_OK;
}

static void all_sizes(c2gpu_ctx *ctx) {
  unsigned seed = 1;
  for (size_t n : SIZES) {
    round_trip(ctx, n, seed++);
    file_trip(ctx, n, seed++);
  }
}

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  const int arg = argc > 2 ? std::atoi(argv[2]) : 0;
  {
    Ctx ctx;
    if (what == "sizes") {
      all_sizes(&ctx);
    } else if (what == "pinned") {  // only `arg` slots can be had
      stub::pinned_left = arg;
      all_sizes(&ctx);
      REQUIRE(stub::pinned_live == arg);
      if (arg < 2) REQUIRE(threads_made == 0);
      stub::pinned_left = -1;  // and the others once there is room
      all_sizes(&ctx);
      REQUIRE(stub::pinned_live == c2gpu_ctx::STAGE_SLOTS);
    } else if (what == "threads") {  // only `arg` threads can be had
      for (size_t n : SIZES) {
        threads_left = arg;
        round_trip(&ctx, n, 3);
        threads_left = arg;
        file_trip(&ctx, n, 4);
      }
    } else if (what == "short") {
      const int fd = temp_file();
      std::vector<char> dev(30 * MIB);
      REQUIRE(ftruncate(fd, 30 * MIB - 1) == 0);
      std::string msg;
      try {
        file_in(&ctx, dev.data(), fd, 0, 30 * MIB, "the file ends early");
      } catch (const Error &e) {
        REQUIRE(e.code == C2GPU_ERR_FORMAT);
        msg = e.msg;
      }
      REQUIRE(msg == "the file ends early");
      close(fd);
      REQUIRE(code_of([&] { file_in(&ctx, dev.data(), -1, 0, 5 * MIB, "short read"); }) == C2GPU_ERR_FORMAT);
      all_sizes(&ctx);
    } else if (what == "null") {
      std::vector<char> a(40 * MIB);
      for (size_t n : {(size_t)1000, a.size()}) {
        REQUIRE(code_of([&] { copy_in(&ctx, a.data(), nullptr, n); }) == C2GPU_ERR_HIP);
        REQUIRE(code_of([&] { copy_in(&ctx, nullptr, a.data(), n); }) == C2GPU_ERR_HIP);
        REQUIRE(code_of([&] { copy_out(&ctx, a.data(), nullptr, n); }) == C2GPU_ERR_HIP);
        REQUIRE(code_of([&] { copy_out(&ctx, nullptr, a.data(), n); }) == C2GPU_ERR_HIP);
      }
      all_sizes(&ctx);
    } else if (what == "full") {
      const int fd = open("/dev/full", O_WRONLY);
      REQUIRE(fd >= 0);
      std::vector<char> dev(30 * MIB);
      REQUIRE(code_of([&] { file_out(&ctx, fd, 0, dev.data(), dev.size()); }) == C2GPU_ERR_FORMAT);
      close(fd);
      all_sizes(&ctx);
    } else if (what == "hip" || what == "throw") {  // the copy after `arg` fails, or throws
      std::vector<char> a(40 * MIB), b(40 * MIB);
      stub::copies_throw = what == "throw";
      const int fd = temp_file();
      for (int q = 0; q < 3; q++) {
        stub::copies_left = arg;
        const int rc = guarded(&ctx, [&] {
          if (q == 0) copy_in(&ctx, a.data(), b.data(), a.size());
          if (q == 1) copy_out(&ctx, a.data(), b.data(), a.size());
          if (q == 2) file_out(&ctx, fd, 0, b.data(), b.size());
        });
        REQUIRE(rc != C2GPU_OK && !ctx.err.empty());
        if (what == "throw") REQUIRE(ctx.err.find("planted") != std::string::npos);
        stub::copies_left = -1;
      }
      all_sizes(&ctx);
    } else if (what == "two") {  // two contexts at once, the slots of each its own
      Ctx other;
      std::thread t([&] { all_sizes(&other); });
      all_sizes(&ctx);
      t.join();
      REQUIRE(stub::pinned_live == 2 * c2gpu_ctx::STAGE_SLOTS);
    } else if (what == "shared") {  // batch workers: at once, on the slots of one context
      Ctx a, b, c;
      a.stage_of = b.stage_of = c.stage_of = &ctx;
      std::thread ta([&] { all_sizes(&a); }), tb([&] { all_sizes(&b); }), tc([&] { all_sizes(&c); });
      all_sizes(&ctx);
      ta.join();
      tb.join();
      tc.join();
      REQUIRE(stub::pinned_live == c2gpu_ctx::STAGE_SLOTS && !a.stage[0].ptr && !b.stage[0].ptr && !c.stage[0].ptr);
    } else {
      return 2;
    }
  }
  REQUIRE(stub::pinned_live == 0);
  std::printf("ok\n");
  return 0;
}
