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
    const int rc = rtt::slab_symbolic(a, &w, rtt::SlabTasks{}, nullptr, 0, nullptr, longest);
    expect(rc == RTT_ERR_OOM, "cursors of 2^40 slots are refused");
    expect(w.slab_cursor_stride <= static_cast<int64_t>(w.slab_cursors.bytes / sizeof(int2)),
           "the cursor stride fits the buffer held");
}

} // namespace

int main()
{
    cursors_after_a_failed_allocation();
    return failures ? 1 : 0;
}
