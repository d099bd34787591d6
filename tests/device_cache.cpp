// Checks of DeviceCache (csrc/device_cache.h); exits 0 if all hold.
#include <cstdio>
#include <thread>
#include <vector>

#include "device_cache.h"

static int failed = 0;

static void check(bool ok, const char* what)
{
    if (!ok) {
        std::printf("failed: %s\n", what);
        failed = 1;
    }
}

int main()
{
    {
        static sph::DeviceCache<4> c;
        std::vector<int> asked(8, 0);
        const auto q = [&](int d) {
            ++asked[d];
            return 1000 + d;
        };
        for (int rep = 0; rep < 3; ++rep)
            for (int d = 0; d < 4; ++d) check(c.get(d, 7, q) == 1000 + d, "each device its own value");
        for (int d = 0; d < 4; ++d) check(asked[d] == 1, "asked once per device");
        check(c.get(6, 7, q) == 1006 && c.get(6, 7, q) == 1006 && asked[6] == 2, "ids past the table");
        check(c.get(-1, 7, [](int) { return 0; }) == 7, "no device");
    }
    {
        static sph::DeviceCache<2> c;
        int n = 0;
        const auto q = [&](int) { return ++n == 1 ? 0 : 42; };
        check(c.get(1, 7, q) == 7, "fallback of a failed query");
        check(c.get(1, 7, q) == 42, "which is made again");
        check(c.get(1, 7, q) == 42 && n == 2, "and then kept");
    }
    {
        static sph::DeviceCache<8> c;
        std::vector<std::thread> t;
        std::atomic<int> bad{0};
        for (int k = 0; k < 8; ++k)
            t.emplace_back([&] {
                for (int i = 0; i < 10000; ++i)
                    if (c.get(i % 8, 7, [](int d) { return d + 1; }) != i % 8 + 1) ++bad;
            });
        for (auto& x : t) x.join();
        check(bad == 0, "several threads");
    }
    return failed;
}
