// Host-side checks of scratch sizes, linked against the library.  Run where
// device allocations fail (no GPU, or sizes no GPU holds): nothing is launched.
#include <cstdio>
#include <cstring>

#include "core.hpp"

namespace {

int failures = 0;

void expect(bool ok, const char *what)
{
    if (!ok) {
        std::printf("FAILED: %s\n", what);
        ++failures;
    }
}

// An allocation of the slab rows' cursors that fails leaves no stride behind:
// the next call would take the buffer for large enough.
void cursors_after_a_failed_allocation()
{
    rtt::SpgemmWork w;
    rtt::DevTiles a;
    const int64_t longest = int64_t(1) << 40;
    const int rc = rtt::slab_symbolic(a, a, &w, rtt::SlabTasks{}, nullptr, 0, nullptr,
                                      rtt::SlabSizes{longest, 1, 1, 1});
    expect(rc == RTT_ERR_OOM, "cursors of 2^40 slots are refused");
    expect(w.slab_cursor_stride <= static_cast<int64_t>(w.slab_cursors.bytes / sizeof(int2)),
           "the cursor stride fits the buffer held");
}

// A hub row's cursors for every workgroup may not fit: fewer workgroups then.
void cursors_of_long_rows()
{
    const size_t gib = size_t(1) << 30;
    const unsigned all = rtt::slab_cursor_blocks(1024, 0, 288 * gib);
    expect(all >= 256, "short rows: every workgroup");
    for (int64_t longest : {int64_t(1) << 20, int64_t(1) << 24, int64_t(1) << 27, int64_t(1) << 30})
        for (size_t free_bytes : {size_t(0), gib, 20 * gib, 288 * gib}) {
            const unsigned n = rtt::slab_cursor_blocks(longest, 0, free_bytes);
            expect(n >= 1 && n <= all, "a workgroup at least, the full grid at most");
            expect(n == 1 || n * static_cast<size_t>(longest) * sizeof(int2) <= free_bytes / 4,
                   "cursors within a quarter of the free memory");
        }
    expect(rtt::slab_cursor_blocks(int64_t(1) << 24, 16 * gib, gib) > 100, "held memory counts");
}

// Positions are ints: a buffer with room for more entries than INT_MAX does
// not count as such (the tile build would write at negative positions).
void entries_of_large_buffers()
{
    const size_t most = INT_MAX;
    expect(rtt::entries_held(0, 8, 1) == -1, "nothing held");
    expect(rtt::entries_held(256, 8, 1) == 31, "a small buffer");
    expect(rtt::entries_held((most + 1) * 8, 8, 1) == INT_MAX, "INT_MAX slots and the zero");
    for (size_t bytes : {(most + 2) * 8, (most + 1) * 9, size_t(1) << 36})
        expect(rtt::entries_held(bytes, 8, 1) == INT_MAX, "larger buffers");
}

} // namespace

int main()
{
    cursors_after_a_failed_allocation();
    cursors_of_long_rows();
    entries_of_large_buffers();
    return failures ? 1 : 0;
}
