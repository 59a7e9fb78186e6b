// in_pieces (tdyn_host.hpp) when memory runs out as its threads start, and when
// a piece throws on a thread: every index is done once or again, none is left,
// and nothing ends the program.
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <new>

static std::atomic<long> fail_at{-1}, allocated{0};
void* operator new(std::size_t n) {
    const long k = fail_at.load();
    if (k >= 0 && allocated++ == k) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

#include "../simbody_amd/csrc/tdyn_host.hpp"

int main() {
    const int n = 100;
    std::atomic<int> done[n];
    int bad = 0;
    for (long k = -1; k < 12; ++k) {
        for (auto& d : done) d = 0;
        allocated = 0;
        fail_at = k;
        tdyn::host::in_pieces(n, 1 << 20, [&](int i0, int i1) { for (int i = i0; i < i1; ++i) ++done[i]; });
        fail_at = -1;
        for (auto& d : done) bad += d < 1;
    }
    for (int t = 0; t < 4; ++t) {
        for (auto& d : done) d = 0;
        std::atomic<int> thrown{0};
        const auto here = std::this_thread::get_id();
        tdyn::host::in_pieces(n, 1 << 20, [&](int i0, int i1) {
            if (std::this_thread::get_id() != here && thrown++ < t) throw 1;
            for (int i = i0; i < i1; ++i) ++done[i];
        });
        for (auto& d : done) bad += d < 1;
    }
    std::printf("%d left\n", bad);
    return bad ? 1 : 0;
}
