// Drives jitnn_amd/csrc/scratch.h with an allocator that keeps books (no GPU).  Prints the name of each check; exit status 0: all hold.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "scratch.h"

static std::map<void *, size_t> live;  // address -> bytes
static size_t room = (size_t)1 << 40;  // bytes the "device" has
static bool refuse_release = false;
static int releases = 0;

struct BookMem {
    static size_t used() {
        size_t u = 0;
        for (auto &b : live) u += b.second;
        return u;
    }
    static void *alloc(size_t bytes) {
        if (used() + bytes > room) return nullptr;
        static size_t next = 0x1000;
        void *p = (void *)next;
        next += bytes;
        live[p] = bytes;
        return p;
    }
    static bool release(void *p) {
        if (refuse_release) return false;
        if (!live.erase(p)) abort();  // freed twice
        ++releases;
        return true;
    }
};
using Block = jitnn::ScratchBlock<BookMem>;
constexpr size_t MiB = (size_t)1 << 20;

#define CHECK(e)                                                       \
    do {                                                               \
        if (!(e)) {                                                    \
            printf("%s:%d: %s does not hold\n", __FILE__, __LINE__, #e); \
            exit(1);                                                   \
        }                                                              \
    } while (0)

static void fresh() {
    live.clear();
    room = (size_t)1 << 40;
    refuse_release = false;
    releases = 0;
}

static void grows_and_reuses() {
    fresh();
    Block b;
    bool waited = false;
    void *p = b.get(3 * MiB + 1, false, &waited);
    CHECK(p && b.capacity() == 4 * MiB && !waited);
    CHECK(b.get(4 * MiB, false, &waited) == p && b.growths() == 1);
    void *q = b.get(5 * MiB, false, &waited);
    CHECK(q && q != p && waited && live.size() == 1 && live.count(q) && b.retired_bytes() == 0);
    b.release_all();
    CHECK(live.empty() && b.capacity() == 0);
}

// A graph records an address; a later eager call needs more.  The recorded block must still be allocated, and new work must
// not be given it.
static void recorded_block_outlives_growth() {
    fresh();
    Block b;
    bool waited = false;
    void *p = b.get(32 * MiB, false, &waited);
    CHECK(b.get(32 * MiB, true, &waited) == p);  // recorded
    void *q = b.get(150 * MiB, false, &waited);
    CHECK(q && q != p && !waited && live.count(p) && live.count(q) && b.retired_bytes() == 32 * MiB);
    CHECK(b.get(32 * MiB, false, &waited) == q);
    void *r = b.get(200 * MiB, false, &waited);  // q was never recorded
    CHECK(r && waited && !live.count(q) && live.count(p));
    b.release_all();
    CHECK(live.empty() && b.retired_bytes() == 0);
}

// Recording at every size: what is kept for graphs stays below what is in use.
static void retired_blocks_are_bounded() {
    fresh();
    Block b;
    bool waited = false;
    for (size_t s = 1; s <= 300; ++s) {
        CHECK(b.get(s * MiB, true, &waited));
        CHECK(b.retired_bytes() < b.capacity());
    }
    b.release_all();
    CHECK(live.empty());
    // where twice the size is not to be had, what the call needs is enough
    room = 100 * MiB;
    CHECK(b.get(40 * MiB, true, &waited) && b.get(60 * MiB, false, &waited));
    CHECK(b.capacity() == 60 * MiB && b.retired_bytes() == 40 * MiB);
    b.release_all();
    CHECK(live.empty());
}

// An address that the runtime would not take back (a capture forbids it) is kept too, and given back later.
static void refused_release_is_not_lost() {
    fresh();
    Block b;
    bool waited = false;
    void *p = b.get(MiB, false, &waited);
    refuse_release = true;
    void *q = b.get(2 * MiB, false, &waited);
    CHECK(q && q != p && !waited && live.size() == 2);
    refuse_release = false;
    b.release_all();
    CHECK(live.empty());
}

int main() {
#define RUN(f) (f(), printf(#f "\n"))
    RUN(grows_and_reuses);
    RUN(recorded_block_outlives_growth);
    RUN(retired_blocks_are_bounded);
    RUN(refused_release_is_not_lost);
    return 0;
}
