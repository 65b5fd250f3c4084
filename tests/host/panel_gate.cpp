// Factorisations in threads: those that fit together run together, the places held never exceed
// the device's, a large one gets its turn among small ones, and errors give places back.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

#include "panel_gate.h"

using namespace bh;

int main()
{
    constexpr long long kCapacity = 512;
    PanelGate gate;
    std::atomic<long long> held{0}, most{0};
    std::atomic<int> together{0}, peak{0}, over{0}, done{0};
    auto factor = [&](long long groups, int times) {
        for (int t = 0; t < times; ++t) {
            try {
                PanelPlaces places;
                places.take(gate, groups, kCapacity);
                const long long h = held += groups;
                const int k = ++together;
                if (h > kCapacity) ++over;
                for (long long m = most; h > m && !most.compare_exchange_weak(m, h);) {}
                for (int m = peak; k > m && !peak.compare_exchange_weak(m, k);) {}
                std::this_thread::sleep_for(std::chrono::microseconds(200));
                --together;
                held -= groups;
                if (t % 7 == 3) throw 1;   // a failed factorisation
            } catch (int) {
            }
        }
        ++done;
    };
    std::vector<std::thread> th;
    for (long long groups : {8, 69, 69, 157, 300, 391, 512}) th.emplace_back(factor, groups, 60);
    for (std::thread &t : th) t.join();
    if (over) return std::printf("%d times more than fit\n", over.load()), 1;
    if (peak < 2) return std::printf("never two together\n"), 1;
    if (done != 7 || held != 0) return std::printf("places left over\n"), 1;
    PanelPlaces all;
    all.take(gate, kCapacity, kCapacity);   // everything was given back
    return 0;
}
