// Host-side check of the shared matrices (pool.hpp): made once, two keys at the
// same time, bounded, and made anew after a failure.
#include "pool.hpp"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <stdexcept>
#include <thread>
#include <vector>

using namespace sphstk;
typedef std::vector<double> Vec;

static int fails = 0;
static void check(bool ok, const char *what) {
    std::printf("%s: %s\n", what, ok ? "ok" : "FAIL");
    fails += !ok;
}

int main() {
    using namespace std::chrono_literals;
    {
        // each of two makers waits (at most 10 s) until the other one is making
        Pool<int, Vec> pool(1 << 20);
        Tables<int, Vec> tab;
        std::atomic<int> in{0}, in2{0}, met{0}, made{0};
        auto meet = [&](std::atomic<int> &n) {
            n++;
            for (int k = 0; k < 1000 && n < 2; k++) std::this_thread::sleep_for(10ms);
            if (n == 2) met++;
        };
        std::vector<std::thread> th;
        for (int t = 0; t < 8; t++)
            th.emplace_back([&, t] {
                const int key = t % 2;
                auto v = pool.get(key, [&] {
                    made++;
                    meet(in);
                    return Vec(10, key);
                });
                const Vec &w = tab.get(key, [&] {
                    made++;
                    meet(in2);
                    return std::make_unique<Vec>(10, key);
                });
                if ((*v)[3] != key || w[3] != key) made += 100;
            });
        for (auto &t : th) t.join();
        check(met == 4, "two keys are made at the same time");
        check(made == 4, "each key is made once for all threads");
    }
    {
        Pool<int, Vec> pool(8 * 1000);
        int made = 0;
        auto get = [&](int key) {
            return pool.get(key, [&] {
                made++;
                return Vec(300, key);
            });
        };
        auto first = get(0);
        get(1), get(2);
        check(pool.bytes() == 7200 && made == 3, "three of 2400 bytes fit 8000");
        get(0);
        get(3); // the least recently used of 0, 1, 2 is 1
        check(pool.bytes() == 7200 && made == 4, "the bound holds");
        get(0), get(2), get(3);
        check(made == 4, "the least recently used one was given back");
        get(1);
        check(made == 5 && pool.bytes() <= 8000, "and is made again when wanted");
        for (int k = 10; k < 20; k++) get(k);
        check((*first)[299] == 0.0, "a holder keeps its value");
        auto big = pool.get(99, [] { return Vec(5000, 1.0); });
        check(big->size() == 5000 && pool.bytes() == 40000, "one value beyond the bound stands alone");
    }
    {
        Pool<int, Vec> pool(1000);
        int tries = 0;
        auto make = [&]() -> Vec {
            if (tries++ == 0) throw std::runtime_error("x");
            return Vec(1, 7.0);
        };
        bool threw = false;
        try {
            pool.get(5, make);
        } catch (const std::runtime_error &) {
            threw = true;
        }
        check(threw && (*pool.get(5, make))[0] == 7.0, "a failure passes through and the value is made anew");
    }
    return fails ? 1 : 0;
}
