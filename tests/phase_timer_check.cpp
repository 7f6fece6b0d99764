// Host build of the phase timers (cqbem_pool.hpp: PhaseEvents, PhaseTimer) for tests/test_phase_timer.py, on event functions of
// its own that count.  Memory runs out inside a timed scope, and while one begins: the first must go on, the second must
// throw std::bad_alloc where the caller can catch it.
#include "../surfaceonlydeformables_amd/csrc/cqbem_pool.hpp"

#include <cstdio>
#include <cstdlib>
#include <new>

static int live = 0, recorded = 0;
extern "C" {
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)(size_t)(0x1000 + ++live), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return live--, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return recorded++, hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
}

static bool exhausted = false;
void *operator new(std::size_t n) {
    void *p = exhausted ? nullptr : std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }

int main() {
    double ms = 0;
    bool caught = false;
    {
        cqbem::PhaseEvents phases;
        {
            cqbem::PhaseTimer t(nullptr, &ms);
            cqbem::PhaseTimer inner(nullptr, &ms);
            exhausted = true;
        }
        try {
            for (int k = 0; k < 100; k++) cqbem::PhaseTimer t(nullptr, &ms);
        } catch (const std::bad_alloc &) {
            caught = true;
        }
        exhausted = false;
        phases.resolve();
    }
    std::printf("%d %d %d %d\n", caught, ms >= 2.0, live, recorded % 2);
    return 0;
}
