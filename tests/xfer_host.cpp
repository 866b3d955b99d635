// The transfers of bnz_xfer.hip (HostLink) on a stand-in runtime whose stream
// runs late: every route, what each pins, and what the caller may reuse when.
#include <cstdio>
#include <new>
#include <vector>

#include "../bonzo_amd/csrc/bnz_xfer.hip"

using namespace bnz;

// the n-th allocation of this thread fails
static thread_local int fail_new = 0;
void *operator new(size_t n) {
  if (fail_new && --fail_new == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

static int bad = 0;
#define CHECK(x) \
  do { \
    if (!(x)) { \
      printf("line %d: %s\n", __LINE__, #x); \
      ++bad; \
    } \
  } while (0)

struct Arrays {  // rows of a box in pools with other boxes' cells around them
  long rows, len, pitch;
  std::vector<double> host, pool;
  Arrays(long r, long l, long p, double v) : rows(r), len(l), pitch(p), host(r * l), pool(r * p, -1.) {
    for (size_t q = 0; q < host.size(); ++q) host[q] = v + q;
  }
  Seg seg() { return Seg{pool.data(), host.data(), pitch, rows, len}; }
  bool up_ok(double v) const {
    for (long r = 0; r < rows; ++r)
      for (long q = 0; q < pitch; ++q)
        if (pool[r * pitch + q] != (q < len ? v + r * len + q : -1.)) return false;
    return true;
  }
};

// several uploads in flight, the host arrays overwritten at once, and back
static void round_trip(HostLink &link, FakeStream &st, long len, bool plain, int many) {
  std::vector<Arrays> w, b;
  for (int k = 0; k < many; ++k) {
    const double v = 1e6 * (k + 1);
    w.emplace_back(plain ? 1 : 9, plain ? 9 * len : len, plain ? 9 * len : len + 7, v);
    b.emplace_back(plain ? 1 : 3, plain ? 3 * len : len, plain ? 3 * len : len + 7, v + 0.5);
  }
  for (int k = 0; k < many; ++k) {
    const Seg s[2] = {w[k].seg(), b[k].seg()};
    CHECK(link.up(0, &st, s, 2) == hipSuccess);
    std::fill(w[k].host.begin(), w[k].host.end(), 0.);
    std::fill(b[k].host.begin(), b[k].host.end(), 0.);
  }
  for (int k = 0; k < many; ++k) {
    const double v = 1e6 * (k + 1);
    const Seg s[2] = {w[k].seg(), b[k].seg()};
    CHECK(link.down(0, &st, s, 2) == hipSuccess);
    CHECK(w[k].up_ok(v) && b[k].up_ok(v + 0.5));
    const Arrays w0(1, 9 * len, 9 * len, v), b0(1, 3 * len, 3 * len, v + 0.5);
    CHECK(w[k].host == w0.host && b[k].host == b0.host);
  }
}

int main() {
  const size_t none = 0, any = ~size_t(0);
  // lengths of the routes: plain copies, the small buffer (up to 1 MB of 96 len
  // bytes), its end, past it, threaded with a short last chunk
  const long lens[] = {3, 600, 1000, 10922, 10923, 30000, 43690, 43691, 200001};
  for (const size_t limit : {any, none, size_t(1) << 20})
    for (const bool plain : {true, false})
      for (const long len : lens) {
        FakeStream st;
        fake.pin_limit = limit;
        fake.launches = fake.copies = 0;
        {
          HostLink link;
          round_trip(link, st, len, plain, len > 30000 ? 2 : 5);
          const size_t bytes = 96 * len, MB = 1u << 20;
          if (limit == none || (plain && bytes < MB / 16) || (bytes > MB && limit != any)) {
            CHECK(fake.launches == 0 && fake.copies > 0 && fake.pinned == 0);  // row by row
          } else {
            CHECK(fake.pinned == (bytes <= MB ? MB : 16 * MB) && fake.launches > 0);
          }
        }
        CHECK(fake.pinned == 0);  // given back
      }
  {  // a small buffer in use grows for a large transfer; one that cannot stays off
    for (const size_t limit : {any, size_t(1) << 20}) {
      FakeStream st;
      fake.pin_limit = limit;
      HostLink link;
      round_trip(link, st, 1000, false, 30);
      CHECK(fake.pinned == size_t(1) << 20);
      Arrays a(1, 2500000, 2500000, 5.);  // in flight: a small upload
      Arrays c(9, 100, 120, 7.);
      const Seg sc = c.seg(), sa = a.seg();
      CHECK(link.up(0, &st, &sc, 1) == hipSuccess);
      CHECK(link.up(0, &st, &sa, 1) == hipSuccess);
      CHECK(fake.pinned == (limit == any ? size_t(16) << 20 : 0));
      round_trip(link, st, 20, false, 3);
      CHECK(a.up_ok(5.) && c.up_ok(7.));
    }
  }
  {  // one segment, nothing to move, download behind queued work
    FakeStream st;
    fake.pin_limit = any;
    HostLink link;
    CHECK(link.up(0, &st, nullptr, 0) == hipSuccess);
    for (const long len : {10L, 20000L}) {
      Arrays a(1, len, len, 3.);
      st.put([&] { std::fill(a.pool.begin(), a.pool.end(), 42.); });
      const Seg s = a.seg();
      CHECK(link.down(0, &st, &s, 1) == hipSuccess);
      CHECK(a.host == std::vector<double>(len, 42.));
    }
  }
  {  // small downloads: a wait and blocking copies, which cost less than two
     // asynchronous ones and a wait
    FakeStream st;
    HostLink link;
    Arrays a(1, 90, 90, 3.), b(1, 30, 30, 4.);
    const Seg s[2] = {a.seg(), b.seg()};
    const long before = st.issued;
    CHECK(link.down(0, &st, s, 2) == hipSuccess && st.issued == before);
  }
  {  // no memory to start the threads with: the caller's moves everything
    FakeStream st;
    HostLink link;
    Arrays a(1, 3000000, 3000000, 6.);
    const Seg s = a.seg();
    CHECK(link.up(0, &st, &s, 1) == hipSuccess);
    std::fill(a.pool.begin(), a.pool.end(), 0.);
    try {
      fail_new = 1;  // a second call's first allocation is its first thread's
      CHECK(link.up(0, &st, &s, 1) == hipSuccess && fail_new == 0);
    } catch (...) {
      CHECK(!"no exception leaves a transfer");
    }
    fail_new = 0;
    CHECK(a.up_ok(6.));
  }
  printf("%d failures\n", bad);
  return bad ? 1 : 0;
}
