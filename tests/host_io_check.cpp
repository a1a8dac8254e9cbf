// Host check of rai_amd/csrc/host_io.h: the copy threads (several callers at
// once, sizes around their blocks) and the bounded block pool (takers past its
// bound, blocks that could not be made, blocks that grow); and of
// raised_limit.h.  Prints "ok", or what is wrong.  Built (also under a thread sanitizer) and run by
// tests/test_cpu_pins.py (test infrastructure only).
#include "host_io.h"
#include "raised_limit.h"

#include <cstdio>
#include <cstdlib>
#include <vector>

namespace {

struct Block {
  int *p = nullptr;
  size_t n = 0;
  int dev = 0;
};

int bad = 0;
void expect(bool ok, const char *what) {
  if (!ok) ++bad, std::printf("wrong: %s\n", what);
}

void copies() {
  const size_t sizes[] = {1, 100, (size_t(1) << 20) - 1, size_t(1) << 20, (size_t(1) << 20) + 1, 3000001};
  std::vector<std::thread> ts;
  std::atomic<int> wrong{0};
  for (int t = 0; t < 4; ++t)
    ts.emplace_back([&, t] {
      for (int it = 0; it < 6; ++it)
        for (size_t n : sizes) {
          std::vector<uint8_t> a(n), b(n, 0);
          for (size_t i = 0; i < n; ++i) a[i] = uint8_t(i * 31 + t + it);
          rai::CopyPool::get().copy(b.data(), a.data(), n);
          if (a != b) ++wrong;
        }
    });
  for (auto &t : ts) t.join();
  expect(wrong == 0, "copies on several threads");
}

using Pool = rai::BoundedPool<Block, 2, 4>;
using Take = rai::PoolTake;

void bounds() {
  static Pool p;
  Block b, c, d;
  static_assert(noexcept(p.give(b)) && noexcept(p.gone(0)), "called from destructors");
  expect(p.take(100, 0, b) == Take::kMake, "first");
  b.n = 100;
  expect(p.take(100, 0, c) == Take::kMake, "second");
  p.gone(0);  // could not be made
  expect(p.take(50, 0, c) == Take::kMake, "second again");
  c.n = 50;
  expect(p.take(1, 0, d) == Take::kNone, "third while two are in use");
  expect(p.take(1, 1, d) == Take::kMake, "another device");
  expect(p.take(1, 4, d) == Take::kNone && p.take(1, -1, d) == Take::kNone, "devices past the table");
  p.give(b);
  p.give(c);
  expect(p.take(40, 0, d) == Take::kBlock && d.n == 50, "the smallest that fits");
  p.give(d);
  expect(p.take(60, 0, d) == Take::kBlock && d.n == 100, "the only one that fits");
  Block e;
  expect(p.take(60, 0, e) == Take::kReplace && e.n == 50, "a small one makes room");
  e.n = 60;
  expect(p.take(1, 0, b) == Take::kNone, "still two");
  p.give(d);
  p.give(e);
  expect(p.take(1000, 0, b) == Take::kReplace && p.take(1000, 0, c) == Take::kReplace, "both grow");
  p.gone(0);
  p.gone(0);
  expect(p.take(1, 0, b) == Take::kMake, "none is left");
}

void kept() {
  static rai::KeptBlocks<Block, 3> k;
  Block b, out;
  static_assert(noexcept(k.keep(b, out)), "called from a destructor");
  expect(!k.take(1, 0, b) && !k.drop(0, b), "nothing kept");
  for (size_t n : {30, 10, 20}) expect(!k.keep(Block{nullptr, n, n == 20}, out), "room");
  expect(k.take(5, 0, b) && b.n == 10, "the smallest that fits, of the device");
  expect(!k.keep(b, out), "back");
  expect(k.keep(Block{nullptr, 40, 0}, out) && out.n == 30, "the oldest leaves");
  expect(!k.take(41, 0, b) && !k.take(1, 2, b), "none fits");
  expect(k.take(11, 0, b) && b.n == 40 && k.drop(0, b) && b.n == 10 && !k.drop(0, b), "of the device only");
  expect(k.take(20, 1, b) && b.n == 20 && !k.take(0, 1, b), "the other device's");
}

// Takers on several threads: a block is never two takers', and there are never
// more than two.
void threads() {
  static Pool p;
  std::atomic<int> live{0}, most{0}, none{0};
  std::vector<std::thread> ts;
  for (int t = 0; t < 6; ++t)
    ts.emplace_back([&, t] {
      for (int it = 0; it < 400; ++it) {
        Block b;
        const size_t n = 1 + (t + it) % 5;
        const Take k = p.take(n, 2, b);
        if (k == Take::kNone) {
          ++none;
          continue;
        }
        if (k == Take::kReplace) std::free(b.p), --live;
        if (k != Take::kBlock) {
          if (it % 17 == 16) {
            p.gone(2);
            continue;
          }
          b = Block{static_cast<int *>(std::calloc(1, sizeof(int))), n, 2};
          const int l = ++live;
          int m = most;
          while (l > m && !most.compare_exchange_weak(m, l)) {
          }
        }
        ++*b.p;  // a race unless the block is this thread's alone
        p.give(b);
      }
    });
  for (auto &t : ts) t.join();
  expect(most <= 2, "blocks at once");
}

// Callers that raise a limit past each other: it never falls, and holds for each
// when its call returns.
void limits() {
  for (int it = 0; it < 200; ++it) {
    rai::RaisedLimit l;
    std::atomic<size_t> set{0};
    std::atomic<int> low{0}, fell{0};
    std::vector<std::thread> ts;
    for (size_t t = 0; t < 4; ++t)
      ts.emplace_back([&, t] {
        for (size_t i = 0; i < 8; ++i) {
          const size_t n = 1 + (3 * i + 5 * t) % 16;
          l.raise(n, [&](size_t b) {
            if (set.exchange(b) >= b) ++fell;
          });
          if (set < n) ++low;
        }
      });
    for (auto &t : ts) t.join();
    expect(low == 0 && fell == 0, "a limit raised on several threads");
  }
}

}  // namespace

int main() {
  copies();
  bounds();
  kept();
  threads();
  limits();
  if (!bad) std::printf("ok\n");
  return bad != 0;
}
