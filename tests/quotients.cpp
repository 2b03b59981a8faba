// The quotients of the kernels that are formed without a division, against the division: test_quotients.py compiles this for the CPU.
// Prints how many differ of all draws' and of those from an approximate reciprocal.
#include <cmath>
#include <cstdio>
#include <thread>
#include <vector>

#include "lbt_internal.h"

namespace {

constexpr int kThreads       = 8;
constexpr uint32_t kDraws    = 2147483646u;  // minstd's draws are 1 .. 2^31 - 2
constexpr uint64_t kSamples  = 4000000;      // a thread and kind of operands

template <typename Work>
uint64_t all_threads(Work work)
{
  std::vector<uint64_t> wrong(kThreads, 0);
  std::vector<std::thread> threads;
  for (int t = 0; t < kThreads; t++) threads.emplace_back([&, t] { wrong[t] = work(t); });
  uint64_t sum = 0;
  for (int t = 0; t < kThreads; t++) {
    threads[t].join();
    sum += wrong[t];
  }
  return sum;
}

struct Random {
  uint64_t s;
  uint64_t next()
  {
    s += 0x9e3779b97f4a7c15ull;
    uint64_t z = s;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
  }
  double unit() { return static_cast<double>(next() >> 11) * 0x1p-53; }
};

bool differs(double n, double d, double e)
{
  return lbt::quotient_from(n, d, (1.0 / d) * (1.0 + e)) != n / d;
}

}  // namespace

int main()
{
  const uint64_t draws = all_threads([](int t) {
    uint64_t wrong = 0;
    const uint32_t from = 1 + static_cast<uint32_t>(static_cast<uint64_t>(kDraws) * t / kThreads);
    const uint32_t to   = 1 + static_cast<uint32_t>(static_cast<uint64_t>(kDraws) * (t + 1) / kThreads);
    for (uint32_t x = from; x < to; x++) wrong += lbt::uniform01(x) != static_cast<double>(x - 1u) / 2147483646.0;
    return wrong;
  });
  const uint64_t quotients = all_threads([](int t) {
    Random r{static_cast<uint64_t>(t) + 1};
    uint64_t wrong = 0;
    for (uint64_t i = 0; i < kSamples; i++) {
      const double e = (2.0 * r.unit() - 1.0) * 0x1p-23;
      // sums of rounded gradients and hessians over their scales, as the gains have them
      const double inv  = std::ldexp(1.0 + r.unit(), static_cast<int>(r.next() % 80) - 60);
      const double grad = static_cast<double>(static_cast<int64_t>(r.next() >> (29 + r.next() % 30))) * inv;
      const double hess = static_cast<double>(static_cast<int64_t>(r.next() >> (29 + r.next() % 30))) * inv;
      wrong += differs(grad * grad, hess + (r.next() % 2 == 0 ? 1e-5 : 1.0), e);
      // any mantissas, and those at the ends, over the exponents that the kernels admit
      const double n = std::ldexp(1.0 + r.unit(), static_cast<int>(r.next() % 800) - 400);
      const double d = std::ldexp(1.0 + r.unit(), static_cast<int>(r.next() % 400) - 200);
      wrong += differs(n, d, e);
      wrong += differs(n, std::ldexp(2.0 - static_cast<double>(r.next() % 64) * 0x1p-52, static_cast<int>(r.next() % 400) - 200), e);
      wrong += differs(std::ldexp(1.0 + static_cast<double>(r.next() % 64) * 0x1p-52, static_cast<int>(r.next() % 400) - 200), d, e);
      // quotients next to the middle of two numbers
      const double q = 1.0 + r.unit();
      wrong += differs(std::fma(q, d, d * 0x1p-53), d, e);
    }
    return wrong;
  });
  std::printf("%llu %llu\n", static_cast<unsigned long long>(draws), static_cast<unsigned long long>(quotients));
  return 0;
}
