// columns_pinned over a made-up address space: bytes [1000, 2000) and [3000, 4000) and [4000, 4500) are pinned
// allocations, everything else is ordinary memory. Prints one 0 or 1 per table.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "sph_pinned.hpp"

namespace {

struct Col {
    void* dst;
    int64_t bytes;
};

char* at(uintptr_t a) { return reinterpret_cast<char*>(a); }

sph::PinnedRange range_of(const char* p)
{
    const uintptr_t edges[][2] = {{1000, 2000}, {3000, 4000}, {4000, 4500}};
    for (const auto& e : edges)
        if (p >= at(e[0]) && p < at(e[1])) return {at(e[0]), (int64_t)(e[1] - e[0])};
    return {};
}

}  // namespace

// arguments: first byte and length of each column, a "/" between tables
int main(int argc, char** argv)
{
    std::vector<Col> cols;
    auto answer = [&]() {
        std::printf("%d\n", (int)sph::columns_pinned(cols.data(), (int)cols.size(), range_of));
        cols.clear();
    };
    for (int i = 1; i < argc; ++i) {
        if (argv[i][0] == '/') answer();
        else if (i + 1 < argc) {
            cols.push_back({at((uintptr_t)std::atoll(argv[i])), std::atoll(argv[i + 1])});
            ++i;
        }
    }
    answer();
    return 0;
}
