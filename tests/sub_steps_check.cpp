// Host build of the patch kernel's scheduled updates (cqbem_kernels.hpp: in_sub_steps), for tests/test_sub_steps.py: a wave's
// 64 lanes are 64 threads that nothing but sync() orders.  Lane i adds its value to slot i % 5 in sub-step i / 5; every update
// reads the slot, gives the other lanes time, and writes it.  Prints the 5 slots, which must hold every lane's value.
#include "../surfaceonlydeformables_amd/csrc/cqbem_kernels.hpp"

#include <pthread.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

int main() {
    constexpr int kLanes = 64, kSlots = 5, kSteps = (kLanes + kSlots - 1) / kSlots;
    std::atomic<long long> slot[kSlots];
    for (auto &s : slot) s = 0;
    pthread_barrier_t wave;
    pthread_barrier_init(&wave, nullptr, kLanes);
    std::vector<std::thread> lanes;
    for (int i = 0; i < kLanes; i++)
        lanes.emplace_back([&, i] {
            cqbem::in_sub_steps(kSteps, i / kSlots, [&] { pthread_barrier_wait(&wave); }, [&] {
                const long long v = slot[i % kSlots];
                std::this_thread::sleep_for(std::chrono::milliseconds(2));
                slot[i % kSlots] = v + (i + 1);
            });
        });
    for (auto &t : lanes) t.join();
    pthread_barrier_destroy(&wave);
    for (auto &s : slot) std::printf("%lld ", s.load());
    std::printf("\n");
    return 0;
}
