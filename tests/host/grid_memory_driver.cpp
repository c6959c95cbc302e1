// CPU driver of the host grid build (linon_amd/csrc/grid.cpp) with a limit on the memory it gets, for
// tests/test_grid_rules.py: `grid_memory_driver BYTES` prints whether the grid was built.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>
#include <vector>

#include "grid.hpp"

static std::atomic<size_t> left{~size_t{0} >> 1};

void* operator new(size_t n) {
    size_t have = left.load();
    do {
        if (have < n) throw std::bad_alloc();
    } while (!left.compare_exchange_weak(have, have - n));
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    const uint32_t n = 5000;  // enough faces for the build's threads
    const float xyz[9] = {0, 0, 0, 1, 0, 0, 0, 1, 0};
    std::vector<uint32_t> faces(3 * n);
    for (uint32_t i = 0; i < 3 * n; ++i) faces[i] = i % 3;
    linon::GridBuild g;
    std::string err;
    left = std::strtoull(argv[1], nullptr, 10);
    bool built = false;
    try {
        built = linon::build_grid(xyz, 3, faces.data(), n, 32, g, err);
    } catch (const std::bad_alloc&) {
    }
    left = ~size_t{0} >> 1;
    std::printf("%s\n", built ? "built" : "no memory");
    return 0;
}
